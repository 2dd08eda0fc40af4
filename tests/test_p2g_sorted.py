"""The sorted form of the phase P2G (mpm_p2g_ws with scratch memory) against
the direct scatter (mpm_p2g, pinned to the FP64 oracle by the phase tests) and
against the oracle itself."""
import ctypes as ct

import numpy as np
import pytest
import torch

from femflow_amd import _lib
from femflow_amd.solvers.mpm import _phase
from oracle import mpm_oracle as O


def _workspace(prm, n):
    b = ct.c_int64()
    _lib.check(_lib.load().mpm_p2g_workspace_bytes(ct.byref(prm), n, ct.byref(b)))
    return b.value


def test_workspace_rule():
    """Scratch is asked for where the sorted form runs, and never where its
    32-bit keys cannot hold the grid."""
    prm3, prm2 = _phase.make_params(3, 64), _phase.make_params(2, 64)
    assert _workspace(prm3, 4095) == 0 and _workspace(prm3, 4096) >= 24 * 4096
    assert _workspace(prm2, 24575) == 0 and _workspace(prm2, 24576) >= 24 * 24576
    assert _workspace(_phase.make_params(3, 1600), 10 ** 6) > 0
    assert _workspace(_phase.make_params(3, 1700), 10 ** 6) == 0


def _particles(n, dim, res, spread, seed, dtype, dev):
    rng = np.random.default_rng(seed)
    x = 0.5 + spread * (rng.random((n, dim)) - 0.5)
    x[:: max(1, n // 7)] = -0.2  # stencils off the grid
    x[1] = np.nan
    eye = np.eye(dim)
    t = lambda a: torch.tensor(a, dtype=dtype, device=dev)  # noqa: E731
    return _phase.StagedParticles(
        t(x), t(rng.normal(size=(n, dim))), t(eye + 0.1 * rng.normal(size=(n, dim, dim))),
        t(rng.normal(size=(n, dim, dim))), t(1 + 0.1 * rng.random((n, 1))), t(0.5 + rng.random(n)),
        t(1e3 * rng.random(n)), t(1e3 * rng.random(n)))


def _p2g(sp, prm, dim, r1, size, dev):
    p, L = sp.struct(), _lib.load()
    gv = torch.zeros(r1 ** dim * dim, dtype=sp.dtype, device=dev)
    gm = torch.zeros(r1 ** dim, dtype=sp.dtype, device=dev)
    oob = torch.zeros(1, dtype=torch.int64, device=dev)
    work = torch.empty(max(size, 1), dtype=torch.uint8, device=dev)
    _lib.check(L.mpm_p2g_ws(torch.cuda.current_stream().cuda_stream, ct.byref(prm), ct.byref(p), _lib.MPM_SNOW, 1.0,
                            None, 0, gv.data_ptr(), gm.data_ptr(), oob.data_ptr(), work.data_ptr(), size))
    return gv.double(), gm.double(), int(oob)


def _rounding_of_additions(sp64, prm, dim, res):
    """Error (2-norm) of adding FP64 contributions to FP32 grids one by one, in
    particle order: (momentum, mass)."""
    host = lambda t: t.tensor.cpu().numpy()  # noqa: E731
    x = host(sp64.x)
    s = x * res - 0.5
    ok = np.all((s > -1) & (s < res - 1), axis=1)  # NaN fails
    args = [host(a)[ok] for a in (sp64.x, sp64.v, sp64.F, sp64.C, sp64.Jp, sp64.mass, sp64.mu0, sp64.lam0)]
    grids = []
    for dtype in (np.float64, np.float32):
        gv, gm = np.zeros((res + 1,) * dim + (dim,), dtype), np.zeros((res + 1,) * dim, dtype)
        O.p2g(*args, O.SNOW, 1.0, float(res), 1.0 / res, 1e-4, 1e-4, gv, gm, check_oob=False)
        grids.append((gv, gm))
    return [float(np.linalg.norm(b.astype(np.float64) - a)) for a, b in zip(*grids)]


@pytest.mark.gpu
@pytest.mark.parametrize("dim,n,res,spread", [
    (3, 4096, 32, 0.2),     # the smallest sorted call, many particles per cell
    (3, 4097, 90, 0.9),     # a remainder, stencil boxes larger than the arena
    (3, 50_003, 20, 0.02),  # every particle in a few cells
    (2, 24_576, 128, 0.3),
    (2, 30_001, 300, 0.95),
])
def test_sorted_equals_direct(gpu, dim, n, res, spread):
    """FP64: equal to rounding (the phase functions' bar, 1e-12 of the grid's
    largest value).  FP32: as near the FP64 sums of the same particles as a
    scatter particle by particle, up to a factor 2 and one rounding of the
    largest value.  That scatter's error: the contributions' own rounding, from
    the form without scratch memory (which sums a workgroup's particles in
    FP64), and one FP32 rounding per addition (_rounding_of_additions)."""
    prm, r1 = _phase.make_params(dim, res, float(res), 1.0 / res, 1e-4, 1e-4), res + 1
    nbytes, off = _workspace(prm, n), len(range(0, n, max(1, n // 7)))
    assert nbytes > 0
    sp = _particles(n, dim, res, spread, n, torch.float32, gpu)
    up = lambda t: t.tensor.double()  # noqa: E731
    sp64 = _phase.StagedParticles(*(up(t) for t in (sp.x, sp.v, sp.F, sp.C, sp.Jp, sp.mass, sp.mu0, sp.lam0)))
    exact, sort64 = (_p2g(sp64, prm, dim, r1, size, gpu) for size in (0, nbytes))
    direct, sort32 = (_p2g(sp, prm, dim, r1, size, gpu) for size in (0, nbytes))
    assert exact[2] == sort64[2] == direct[2] == sort32[2] == off + 1
    adds = _rounding_of_additions(sp64, prm, dim, res)
    for e, s64, d, s32, a in zip(exact[:2], sort64[:2], direct[:2], sort32[:2], adds):
        top = float(e.abs().max())
        assert float((s64 - e).abs().max()) <= 1e-12 * top
        assert float((s32 - e).norm()) <= 2 * np.hypot(float((d - e).norm()), a) + 1.2e-7 * top


@pytest.mark.gpu
def test_sorted_matches_oracle(gpu):
    """three_d.p2g above the line (sorted) against the NumPy oracle."""
    from femflow_amd.solvers.mpm import three_d
    from femflow_amd.solvers.mpm.particle import ParticleSet

    n = 6000
    st, pr = O.scene_3d_cubes(n=n, res=32, seed=5)
    st["v"] = st["v"] + np.random.default_rng(1).normal(size=st["v"].shape)
    r1 = pr["res"] + 1
    gv, gm = np.zeros((r1, r1, r1, 3)), np.zeros((r1, r1, r1, 1))
    O.p2g_3d(pr["inv_dx"], 1.0, pr["dx"], pr["dt"], pr["volume"], gv, gm, st["x"], st["mass"], st["mu0"], st["lam0"],
             st["v"], st["F"], st["C"], st["Jp"])
    t = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device=gpu)  # noqa: E731
    got_v, got_m = t(np.zeros_like(gv)), t(np.zeros_like(gm))
    ps = ParticleSet(t(st["x"]), t(st["mass"]), t(st["mu0"]), t(st["lam0"]))
    three_d.p2g(pr["inv_dx"], 1.0, pr["dx"], pr["dt"], pr["volume"], got_v, got_m, ps, t(st["v"]), t(st["F"]),
                t(st["C"]), t(st["Jp"]))
    for a, b in ((gv, got_v), (gm, got_m)):
        assert np.abs(a - b.cpu().numpy()).max() <= 1e-12 * np.abs(a).max()
