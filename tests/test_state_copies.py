"""Upload and download of the engine's state: every path a state can take
between them (records, tiles, one and two passes) keeps every value."""
import numpy as np
import pytest
import torch

from femflow_amd.engine import Engine, MaterialSpec, SceneSpec

KEYS = ("x", "v", "F", "C", "Jp")


def _state(n, dev, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    r = lambda *s: torch.rand(*s, generator=g, device=dev)  # noqa: E731
    s = dict(x=0.3 + 0.4 * r(n, 3), v=r(n, 3) - 0.5, F=torch.eye(3, device=dev) + 0.01 * (r(n, 3, 3) - 0.5),
             C=r(n, 3, 3) - 0.5, Jp=0.9 + 0.2 * r(n), mass=1e-3 * (0.5 + r(n)), mu0=1e3 * r(n), lam0=1e3 * r(n),
             material=(3 * r(n)).int(), scene=(2 * r(n)).int())
    return s


def _engine(n, scenes=1):
    return Engine([SceneSpec(res=32 + i, dt=1e-5, volume=1e-3) for i in range(scenes)],
                  [MaterialSpec("elastic"), MaterialSpec("snow", 10.0), MaterialSpec("water")], n_max=n)


def _upload(eng, s, scene=None):
    eng.upload(*(s[k] for k in KEYS), s["mass"], s["mu0"], s["lam0"], s["material"], scene)


def _download(eng, s):
    out = {k: torch.full_like(s[k], float("nan")) for k in KEYS}
    eng.download(*(out[k] for k in KEYS))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, (1 << 20) - 1, (1 << 20) + 65])
def test_round_trip_without_a_run(gpu, n):
    s = _state(n, gpu)
    eng = _engine(n)
    _upload(eng, s)
    assert torch.equal(eng.positions(), s["x"])
    for _ in range(2):  # straight from the records, then from the tiles
        out = _download(eng, s)
        assert all(torch.equal(out[k], s[k]) for k in KEYS)
    m = s["mass"].double()
    want = torch.cat((m.sum()[None], (m[:, None] * s["v"].double()).sum(0), (m[:, None] * s["x"].double()).sum(0)))
    _upload(eng, s)  # the sums read the records too
    assert np.allclose(eng.particle_sums(), want.cpu().numpy(), rtol=1e-9, atol=1e-12 * n)
    eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,scenes,graph", [(5000, 1, True), (5003, 2, True), (70_001, 1, False)])
def test_run_from_records_equals_run_from_tiles(gpu, n, scenes, graph):
    """A run right after the upload moves the particles out of the records; a
    download in between puts them into tiles first.  Same arithmetic, so the
    same state; a second upload replays the captured graphs."""
    s = _state(n, gpu, seed=n)
    scene = s["scene"] if scenes == 2 else None
    eng = _engine(n, scenes)
    eng.tune(use_graph=graph)
    outs = []
    for between in (False, True, False, True):
        _upload(eng, s, scene)
        if between:
            _download(eng, s)
        eng.run(3)
        outs.append(_download(eng, s))
    for o in outs[1:]:
        for k in KEYS:
            assert torch.equal(o[k], outs[0][k]), k
    assert not torch.equal(outs[0]["x"], s["x"])
    eng.close()


@pytest.mark.gpu
def test_two_pass_download_after_runs(gpu):
    """Both buffer parities, a state above the two-pass line: what comes down
    equals what a second engine with the same history holds in one pass
    (its particle positions), and a further run is not disturbed by the
    scratch use of the other state copy."""
    n = (1 << 20) + 3
    s = _state(n, gpu, seed=9)
    eng, ref = _engine(n), _engine(n)
    for e in (eng, ref):
        _upload(e, s)
    for _ in range(2):
        for e in (eng, ref):
            e.request_rebin()
            e.run(2)
        out = _download(eng, s)
        assert torch.equal(out["x"], ref.positions())
        assert all(bool(torch.isfinite(out[k]).all()) for k in KEYS)
    eng.close()
    ref.close()


@pytest.mark.gpu
def test_states_of_deferred_particles(gpu):
    """Per-substep states are written after the grid update that finishes the
    FP64-deferred particles: with 600 near-degenerate ones (snow for the G2P
    side, elastic for the P2G side) every recorded substep agrees with a run
    that ends there, to the order of their float atomics (1e-5 of the largest
    value, 1e-4 for C, which carries 1 / dx)."""
    n, k = 20_000, 4
    s = _state(n, gpu, 3)
    g = torch.Generator(device=gpu).manual_seed(9)
    q = torch.linalg.qr(torch.randn(600, 3, 3, generator=g, device=gpu))[0]
    q = q * torch.sign(torch.linalg.det(q))[:, None, None]
    s["material"].fill_(0)
    s["material"][300:600] = 1
    s["F"][:300] = q[:300] * torch.tensor([1.02, 0.98, 2e-4], device=gpu)
    s["F"][300:600] = q[300:] * torch.tensor([1.0, 0.95, 0.004], device=gpu)
    s["mu0"].fill_(300.0)
    s["lam0"].fill_(200.0)
    eng = _engine(n)
    eng.tune(sort_every=3)
    _upload(eng, s)
    rec = {f: torch.empty((k,) + tuple(s[f].shape), device=gpu) for f in KEYS}
    eng.run_states(k, *(rec[f] for f in KEYS))
    assert eng.fallback_count() >= 500
    for j in range(k):
        _upload(eng, s)
        eng.run(j + 1)
        got = {f: torch.empty_like(s[f]) for f in KEYS}
        eng.download(*(got[f] for f in KEYS))
        for f in KEYS:
            off = float((rec[f][j] - got[f]).abs().max()) / float(got[f].abs().max())
            assert off <= (1e-4 if f == "C" else 1e-5), (j, f, off)
    eng.close()
