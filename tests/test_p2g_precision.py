"""FP32 rounding of the sorted phase P2G's terms: no more than that of the terms
taken as the reference writes them (three_d/p2g.py:67-80), w (m v + A (n - fx) dx)."""
import ctypes as ct

import numpy as np
import pytest
import torch

from femflow_amd import _lib
from femflow_amd.solvers.mpm import _phase
from oracle import mpm_oracle as O


def _terms_in_fp32(s, dim, res):
    """The grid momentum from terms rounded to FP32 at each operation (without
    stress, A = m C), added up in FP64."""
    f = np.float32
    x, v, C, m = (s[k].astype(f) for k in ("x", "v", "C", "mass"))
    t = x.astype(np.float64) * res - 0.5
    base = t.astype(np.int64)
    fx = (x * f(res) - base.astype(f)).astype(f)
    w = [f(0.5) * (f(1.5) - fx) ** 2, f(0.75) - (fx - f(1)) ** 2, f(0.5) * (fx - f(0.5)) ** 2]
    A, mv, dx = C * m[:, None, None], v * m[:, None], f(1.0 / res)
    out = np.zeros((res + 1,) * dim + (dim,))
    for o in np.ndindex(*(3,) * dim):
        dp = (np.array(o, f) - fx) * dx
        weight, ad = np.ones(len(x), f), np.zeros_like(v)
        for d in range(dim):
            weight = weight * w[o[d]][:, d]
            ad = ad + A[:, :, d] * dp[:, d:d + 1]
        term = (weight[:, None] * (mv + ad)).astype(np.float64)
        np.add.at(out, tuple(base[:, d] + o[d] for d in range(dim)), term)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("dim,n,res,side", [(3, 5000, 64, 0.55), (3, 20_000, 64, 0.2), (2, 30_000, 256, 0.9)])
def test_sorted_terms(gpu, dim, n, res, side):
    """Velocity gradients that make A (n - fx) dx some times m v.  The bar: the
    FP32 terms' error, and one FP32 rounding of each node for the form in which
    it is written."""
    rng = np.random.default_rng(dim)
    s = dict(x=0.5 + side * (rng.random((n, dim)) - 0.5), v=0.1 * rng.normal(size=(n, dim)),
             F=np.broadcast_to(np.eye(dim), (n, dim, dim)), C=40.0 * rng.normal(size=(n, dim, dim)), Jp=np.ones((n, 1)),
             mass=0.5 + rng.random(n), mu0=np.zeros(n), lam0=np.zeros(n))
    t = {k: torch.tensor(np.ascontiguousarray(a), dtype=torch.float32, device=gpu) for k, a in s.items()}
    s = {k: a.double().cpu().numpy() for k, a in t.items()}
    prm, r1 = _phase.make_params(dim, res, float(res), 1.0 / res, 1e-4, 1e-4), res + 1
    sp = _phase.StagedParticles(t["x"], t["v"], t["F"], t["C"], t["Jp"], t["mass"], t["mu0"], t["lam0"])
    gv, gm = torch.zeros((r1,) * dim + (dim,), device=gpu), torch.zeros((r1,) * dim, device=gpu)
    b, p, L = ct.c_int64(), sp.struct(), _lib.load()
    _lib.check(L.mpm_p2g_workspace_bytes(ct.byref(prm), n, ct.byref(b)))
    assert b.value > 0
    work = torch.empty(b.value, dtype=torch.uint8, device=gpu)
    _lib.check(L.mpm_p2g_ws(torch.cuda.current_stream().cuda_stream, ct.byref(prm), ct.byref(p), _lib.MPM_ELASTIC, 1.0,
                            None, 0, gv.data_ptr(), gm.data_ptr(), None, work.data_ptr(), b.value))
    exact, mass = np.zeros((r1,) * dim + (dim,)), np.zeros((r1,) * dim)
    O.p2g(s["x"], s["v"], s["F"], s["C"], s["Jp"], s["mass"], s["mu0"], s["lam0"], O.ELASTIC, 1.0, float(res), 1.0 / res,
          1e-4, 1e-4, exact, mass)
    error = np.linalg.norm(gv.double().cpu().numpy() - exact)
    bar = np.hypot(np.linalg.norm(_terms_in_fp32(s, dim, res) - exact), np.linalg.norm(exact) * 2.0 ** -24)
    print("sorted terms", dim, n, error / bar, flush=True)
    assert error <= bar


@pytest.mark.gpu
def test_2d_forms_round_alike(gpu):
    """Small strains of stiff particles: F - R is most of the error, and it is the
    same function in every form.  The form without scratch memory (the arena, at
    this density) is at most 2% of it further from the exact sums than the sorted
    one."""
    n, res, dim = 30_000, 256, 2
    rng = np.random.default_rng(7)
    side = (n / 4) ** 0.5 / res
    h = dict(x=0.5 + side * (rng.random((n, 2)) - 0.5), v=0.1 * rng.normal(size=(n, 2)),
             F=np.eye(2) + 0.01 * rng.normal(size=(n, 2, 2)), C=np.zeros((n, 2, 2)), Jp=np.ones((n, 1)),
             mass=np.full(n, 1e-6), mu0=np.full(n, 2e3), lam0=np.full(n, 1e3))
    t = {k: torch.tensor(a, dtype=torch.float32, device=gpu) for k, a in h.items()}
    h = {k: a.double().cpu().numpy() for k, a in t.items()}
    prm, r1 = _phase.make_params(dim, res, float(res), 1.0 / res, 1e-4, 1e-6), res + 1
    sp = _phase.StagedParticles(t["x"], t["v"], t["F"], t["C"], t["Jp"], t["mass"], t["mu0"], t["lam0"])
    b, p, L = ct.c_int64(), sp.struct(), _lib.load()
    _lib.check(L.mpm_p2g_workspace_bytes(ct.byref(prm), n, ct.byref(b)))
    work = torch.empty(b.value, dtype=torch.uint8, device=gpu)
    exact, mass = np.zeros((r1, r1, 2)), np.zeros((r1, r1))
    O.p2g(h["x"], h["v"], h["F"], h["C"], h["Jp"], h["mass"], h["mu0"], h["lam0"], O.ELASTIC, 1.0, float(res), 1.0 / res,
          1e-4, 1e-6, exact, mass)
    errors = []
    for size in (0, b.value):
        gv, gm = torch.zeros((r1, r1, 2), device=gpu), torch.zeros((r1, r1), device=gpu)
        _lib.check(L.mpm_p2g_ws(torch.cuda.current_stream().cuda_stream, ct.byref(prm), ct.byref(p), _lib.MPM_ELASTIC,
                                1.0, None, 0, gv.data_ptr(), gm.data_ptr(), None, work.data_ptr(), size))
        errors.append(np.linalg.norm(gv.double().cpu().numpy() - exact))
    print("2D forms", errors, np.linalg.norm(exact), flush=True)
    assert errors[0] <= 1.02 * errors[1]
