"""The entry points behind the phase functions that count, pass constants by
value and bin on a stream: mpm_count_oob and mpm_p2g_uniform against the phase
kernels' own count and per-particle constants, mpm_bin_ws against mpm_bin."""
import ctypes as ct

import numpy as np
import pytest
import torch

from femflow_amd import _lib
from femflow_amd.solvers.mpm import _phase, three_d
from femflow_amd.solvers.mpm.particle import ParticleSet


def _stream():
    return torch.cuda.current_stream().cuda_stream


def test_bad_arguments():
    """Refused before anything is launched."""
    L, prm, one = _lib.load(), _phase.make_params(3, 16, 16.0), ct.c_int64(0)
    p = _lib.Particles(4, _lib.MPM_F32, 0, None, None, None, None, None, None, None, None, None)
    assert L.mpm_count_oob(None, ct.byref(prm), ct.byref(p), ct.addressof(one)) == _lib.MPM_ERR_ARG
    assert L.mpm_p2g_uniform(None, ct.byref(prm), ct.byref(p), -1, 1.0, 1.0, 1.0, 1.0, 8, 8, None,
                             0) == _lib.MPM_ERR_ARG
    need = ct.c_int64()
    assert L.mpm_bin_workspace_bytes(1000, ct.byref(need)) == _lib.MPM_OK and need.value >= 24 * 1000
    assert L.mpm_bin_workspace_bytes(-1, ct.byref(need)) == _lib.MPM_ERR_ARG
    assert L.mpm_bin_ws(None, 3, 16, 16.0, _lib.MPM_KEY_BLOCKED, 16, 1000, 16, 16, 16, need.value - 1) == _lib.MPM_ERR_ARG
    assert L.mpm_bin_ws(None, 3, 4096, 4096.0, _lib.MPM_KEY_BLOCKED, 16, 10, 16, 16, 16, 1 << 20) == _lib.MPM_ERR_ARG


@pytest.mark.gpu
@pytest.mark.parametrize("dim", (2, 3))
@pytest.mark.parametrize("dtype", (torch.float32, torch.float64))
@pytest.mark.parametrize("n", (1, 64, 257, 5000))
def test_count_agrees_with_the_phases(gpu, dim, dtype, n):
    """Positions one rounding on each side of the grid's limits, far off and
    NaN: the count is the phase kernels' own, exactly; constants by value give
    the sums of per-particle ones (same order of additions apart: 1e-5 FP32,
    1e-12 FP64 of the largest)."""
    res, rng, L = 37, np.random.default_rng(n), _lib.load()
    x = rng.random((n, dim)) * 0.8 + 0.1
    edge = np.array([-0.5, res - 0.5]) / res
    near = np.float32 if dtype == torch.float32 else np.float64
    for i in range(0, n, 3):
        e = near(edge[rng.integers(2)])
        x[i, rng.integers(dim)] = [e, np.nextafter(e, near(2)), np.nextafter(e, near(-2)), np.nan, 5.0][rng.integers(5)]
    t = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=dtype, device=gpu)  # noqa: E731
    eye = np.broadcast_to(np.eye(dim), (n, dim, dim))
    full = lambda a: t(np.full(n, a))  # noqa: E731
    sp = _phase.StagedParticles(t(x), t(rng.normal(size=(n, dim))), t(eye), t(0 * eye), t(np.ones((n, 1))), full(0.7),
                                full(300.0), full(200.0))
    prm, r1 = _phase.make_params(dim, res, float(res), 1.0 / res, 1e-4, 1e-4), res + 1
    p = sp.struct()
    grids = [(torch.zeros(r1 ** dim * dim, dtype=dtype, device=gpu), torch.zeros(r1 ** dim, dtype=dtype, device=gpu))
             for _ in range(2)]
    counts = torch.zeros(3, dtype=torch.int64, device=gpu)
    at = lambda i: counts.data_ptr() + 8 * i  # noqa: E731
    (gv, gm), (uv, um) = grids
    _lib.check(L.mpm_count_oob(_stream(), ct.byref(prm), ct.byref(p), at(0)))
    _lib.check(L.mpm_p2g(_stream(), ct.byref(prm), ct.byref(p), 0, 1.0, None, 0, gv.data_ptr(), gm.data_ptr(), at(1)))
    bare = _phase.StagedParticles(sp.x.tensor, sp.v.tensor, sp.F.tensor, sp.C.tensor, sp.Jp.tensor, None, None, None)
    q = bare.struct()
    _lib.check(L.mpm_p2g_uniform(_stream(), ct.byref(prm), ct.byref(q), 0, 1.0, 0.7, 300.0, 200.0, uv.data_ptr(),
                                 um.data_ptr(), None, 0))
    _lib.check(L.mpm_g2p(_stream(), ct.byref(prm), ct.byref(p), 0, 0.0, 0.0, None, 0, gv.data_ptr(), at(2)))
    a, b, c = counts.tolist()
    assert a == b == c
    bar = 1e-5 if dtype == torch.float32 else 1e-12
    for g, u in ((gv, uv), (gm, um)):
        assert float((g - u).abs().max()) <= bar * max(float(g.abs().max()), 1e-30)


@pytest.mark.gpu
def test_phases_raise_and_keep_going(gpu):
    """A particle off the grid is reported by the call that meets it, and the
    others are still moved."""
    n, res = 300, 16
    x = torch.rand(n, 3, dtype=torch.float64, device=gpu) * 0.5 + 0.25
    x[7] = 3.0
    eye = torch.eye(3, dtype=torch.float64, device=gpu).expand(n, 3, 3).contiguous()
    one = torch.ones(n, dtype=torch.float64, device=gpu)
    ps = ParticleSet(x, one, one, one)
    v, F, C, Jp = torch.zeros_like(x), eye.clone(), torch.zeros_like(eye), one.clone().reshape(-1, 1)
    gv = torch.zeros(res + 1, res + 1, res + 1, 3, dtype=torch.float64, device=gpu)
    gm = torch.zeros(res + 1, res + 1, res + 1, 1, dtype=torch.float64, device=gpu)
    with pytest.raises(RuntimeError, match="1 particle"):
        three_d.p2g(float(res), 1.0, 1 / res, 1e-3, 1e-3, gv, gm, ps, v, F, C, Jp)
    assert abs(float(gm.sum()) - (n - 1)) < 1e-9
    gv.fill_(1.0)
    with pytest.raises(RuntimeError, match="1 particle"):
        three_d.g2p(float(res), 1e-3, gv, ps, v, F, C, Jp)
    assert float(v[7].abs().max()) == 0.0 and float((v.sum() / 3 - (n - 1)).abs()) < 1e-9


@pytest.mark.gpu
def test_bin_ws_on_another_stream(gpu):
    """mpm_bin's keys and order, from a stream of the caller's."""
    n, L = 70_001, _lib.load()
    x = torch.rand(n, 3, device=gpu)
    out = torch.empty(4, n, dtype=torch.int32, device=gpu)
    need = ct.c_int64()
    _lib.check(L.mpm_bin_workspace_bytes(n, ct.byref(need)))
    work = torch.empty(need.value, dtype=torch.uint8, device=gpu)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    _lib.check(L.mpm_bin_ws(side.cuda_stream, 3, 64, 64.0, _lib.MPM_KEY_BLOCKED, x.data_ptr(), n, out[0].data_ptr(),
                            out[1].data_ptr(), work.data_ptr(), need.value))
    side.synchronize()
    _lib.check(L.mpm_bin(None, 3, 64, 64.0, _lib.MPM_KEY_BLOCKED, x.data_ptr(), n, out[2].data_ptr(), out[3].data_ptr()))
    assert torch.equal(out[0], out[2]) and torch.equal(out[1], out[3])


@pytest.mark.gpu
@pytest.mark.parametrize("dim,n,res,spread", [
    (2, 1, 40, 0.1),
    (2, 511, 60, 0.5),      # one workgroup, not full
    (2, 513, 60, 0.5),      # a second one of one particle
    (2, 3000, 200, 0.9),    # the arena holds a part of the box
    (3, 255, 20, 0.5),
    (3, 257, 20, 0.5),
    (3, 2000, 60, 0.8),
    (3, 300, 150, 0.9),     # not one layer of it
])
@pytest.mark.parametrize("dtype", (torch.float32, torch.float64))
def test_few_particles_match_oracle(gpu, dim, n, res, spread, dtype):
    """P2G by workgroup boxes against the oracle's FP64 sums: 1e-12 of the
    largest value in FP64; in FP32 2e-6 (some ten roundings of a contribution,
    whose terms reach several times their sum) and 2e-7 res (x / dx rounds by
    up to 6e-8 res cells, on each axis)."""
    from oracle import mpm_oracle as O

    rng, L, r1 = np.random.default_rng(n), _lib.load(), res + 1
    x = 0.5 + spread * (rng.random((n, dim)) - 0.5)
    up = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=dtype, device=gpu)  # noqa: E731
    x, v = up(x), up(rng.normal(size=(n, dim)))
    F = up(np.eye(dim) + 0.02 * rng.normal(size=(n, dim, dim)))
    C, Jp = up(rng.normal(size=(n, dim, dim))), up(np.ones((n, 1)))
    mass, mu, lam = (up(np.full(n, a)) for a in (0.5, 3.0, 2.0))
    sp = _phase.StagedParticles(x, v, F, C, Jp, mass, mu, lam)
    prm = _phase.make_params(dim, res, float(res), 1.0 / res, 1e-4, 1e-4)
    gv = torch.zeros((r1,) * dim + (dim,), dtype=dtype, device=gpu)
    gm = torch.zeros((r1,) * dim, dtype=dtype, device=gpu)
    p = sp.struct()
    _lib.check(L.mpm_p2g(_stream(), ct.byref(prm), ct.byref(p), _lib.MPM_ELASTIC, 1.0, None, 0, gv.data_ptr(),
                         gm.data_ptr(), None))
    host = lambda a: a.double().cpu().numpy()  # noqa: E731
    ev, em = np.zeros(gv.shape), np.zeros(gm.shape + (1,) * (dim == 3))
    args = [host(a) for a in (x, v, F, C, Jp)]
    if dim == 3:
        O.p2g_3d(float(res), 1.0, 1 / res, 1e-4, 1e-4, ev, em, args[0], host(mass), host(mu), host(lam), *args[1:])
    else:
        O.p2g_2d(float(res), 1.0, 3.0, 2.0, 0.5, 1 / res, 1e-4, 1e-4, ev, em, *args)
    bar = 2e-6 + 2e-7 * res if dtype == torch.float32 else 1e-12
    for g, e in ((gv, ev), (gm, em.reshape(gm.shape))):
        assert np.abs(host(g) - e).max() <= bar * np.abs(e).max()
