"""Chunks of at most 128 particles of engines with many scenes run in one wave
each, in a launch of their own: the results are those of engines of one scene,
which run every chunk in the four-wave kernel, to FP32 rounding (another
instance of the same code), and the same from run to run."""
import numpy as np
import pytest
import torch

from femflow_amd.engine import Engine, MaterialSpec, SceneSpec

pytestmark = pytest.mark.gpu
KEYS = ("x", "v", "F", "C", "Jp")


def _state(counts, dev):
    """Scene i: counts[i] particles in one block of 4^3 cells (res 32), at rest
    relative to the block for the few substeps that are run."""
    rng = np.random.default_rng(5)
    n = sum(counts)
    scene = np.repeat(np.arange(len(counts)), counts)
    x = (8 + 0.75 + 3.2 * rng.random((n, 3))) / 32  # bases 8..11 of block (2, 2, 2)
    F = np.eye(3) + 0.003 * rng.normal(size=(n, 3, 3))
    perm = rng.permutation(n)
    t = lambda a, d=torch.float32: torch.tensor(np.ascontiguousarray(a[perm]), dtype=d, device=dev)  # noqa: E731
    return dict(x=t(x), v=t(0.1 * rng.normal(size=(n, 3))), F=t(F), C=t(rng.normal(size=(n, 3, 3))),
                Jp=t(np.ones(n)), mass=t(1e-6 * (0.5 + rng.random(n))), mu0=t(np.full(n, 300.0)),
                lam0=t(np.full(n, 200.0)), material=t(rng.integers(0, 3, n), torch.int32),
                scene=t(scene, torch.int32))


def _run(s, scene, nscenes, splits):
    eng = Engine([SceneSpec(res=32, dt=1e-5, volume=1e-6) for _ in range(nscenes)],
                 [MaterialSpec("elastic"), MaterialSpec("snow", 10.0), MaterialSpec("water")], n_max=len(s["x"]))
    eng.upload(*(s[k] for k in KEYS), s["mass"], s["mu0"], s["lam0"], s["material"], scene)
    for k in splits:
        eng.run(k)
    out = {k: torch.empty_like(s[k]) for k in KEYS}
    eng.download(*(out[k] for k in KEYS))
    assert eng.fallback_count() == 0
    eng.close()
    return out


@pytest.mark.parametrize("counts", [
    (1, 63, 64, 65, 127, 128, 129, 513),  # both sides of a row, of the limit, of a second chunk
    (5,) * 40,                            # small ones only
    (300,) * 8,                           # none
    (0, 700, 0, 0, 0, 0, 0, 0, 2),        # empty scenes
])
@pytest.mark.parametrize("splits", [(1,), (5,), (2, 3)])
def test_small_chunks_equal_the_others(gpu, counts, splits):
    s = _state(counts, gpu)
    run = lambda sel, ids, nscenes: _run(sel, ids, nscenes, splits)  # noqa: E731
    outs = [run(s, s["scene"], len(counts)) for _ in range(2)]
    for k in KEYS:
        assert torch.equal(outs[0][k], outs[1][k]), k
    # scenes of one chunk in both kinds of engine (beyond 256 particles an
    # engine of one scene cuts its blocks elsewhere)
    for i in [i for i, c in enumerate(counts) if 0 < c <= 256][:8]:
        at = torch.nonzero(s["scene"] == i).flatten()
        alone = run({k: a[at].contiguous() for k, a in s.items()}, None, 1)
        for k in KEYS:
            a, b = outs[0][k][at], alone[k]
            # C carries 4 / dx of the velocities' rounding
            assert float((a - b).abs().max()) <= (1e-5 if k == "C" else 1e-6) * float(b.abs().max()), (i, k)
