"""The phase P2G without scratch memory: each of its forms (sums by cell where
lanes share cells, or where nodes get few adds; the arena; the arena's layers that
do not fit) against the oracle."""
import ctypes as ct

import numpy as np
import pytest
import torch

from femflow_amd import _lib
from femflow_amd.solvers.mpm import _phase
from oracle import mpm_oracle as O


def _particles(n, dim, res, ppc, order, seed):
    rng = np.random.default_rng(seed)
    side = min(0.9, (n / ppc) ** (1 / dim) / res)
    x = 0.5 + side * (rng.random((n, dim)) - 0.5)
    if order == "cells":
        b = np.trunc(x * res - 0.5).astype(int)
        x = x[np.lexsort([b[:, d] for d in reversed(range(dim))])]
    if n > 8:
        x[3], x[n // 2] = -0.2, np.nan  # stencils off the grid
    return dict(x=x, v=rng.normal(size=(n, dim)), F=np.eye(dim) + 0.1 * rng.normal(size=(n, dim, dim)),
                C=rng.normal(size=(n, dim, dim)), Jp=np.ones((n, 1)), mass=0.5 + rng.random(n),
                mu0=1e3 * rng.random(n), lam0=1e3 * rng.random(n))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("dim,n,res,ppc,order", [
    (3, 128, 64, 0.05, "any"), (3, 131, 64, 0.05, "any"),   # half a workgroup, and more: arena / sums without one
    (3, 3000, 64, 0.3, "any"), (3, 3000, 64, 2, "any"),     # few and many adds per node
    (3, 9000, 64, 2, "any"),                                # an arena that holds part of the layers
    (3, 1000, 64, 2, "cells"), (3, 1000, 64, 12, "cells"),  # runs of about 2 and of 12 particles
    (3, 30_001, 96, 8, "cells"), (3, 30_001, 96, 0.5, "cells"),
    (3, 4000, 32, 300, "cells"), (3, 1, 8, 1, "any"),
    (2, 256, 128, 0.05, "any"), (2, 260, 128, 0.05, "any"),
    (2, 9000, 256, 0.3, "any"), (2, 9000, 256, 8, "any"), (2, 30_001, 256, 2, "any"),
    (2, 9000, 256, 3, "cells"), (2, 9000, 256, 20, "cells"), (2, 7, 16, 1, "any"),
])
def test_against_the_oracle(gpu, dim, n, res, ppc, order, dtype):
    """FP64: the phase functions' bar, 1e-12 of the largest value.  FP32: the
    roundings of a particle's terms and of a node's additions."""
    host = _particles(n, dim, res, ppc, order, n)
    t = {k: torch.tensor(a, dtype=dtype, device=gpu) for k, a in host.items()}
    prm, r1 = _phase.make_params(dim, res, float(res), 1.0 / res, 1e-4, 1e-4), res + 1
    sp = _phase.StagedParticles(t["x"], t["v"], t["F"], t["C"], t["Jp"], t["mass"], t["mu0"], t["lam0"])
    gv = torch.zeros((r1,) * dim + (dim,), dtype=dtype, device=gpu)
    gm, oob = torch.zeros((r1,) * dim, dtype=dtype, device=gpu), torch.zeros(1, dtype=torch.int64, device=gpu)
    p = sp.struct()
    _lib.check(_lib.load().mpm_p2g(torch.cuda.current_stream().cuda_stream, ct.byref(prm), ct.byref(p),
                                   _lib.MPM_ELASTIC, 1.0, None, 0, gv.data_ptr(), gm.data_ptr(), oob.data_ptr()))
    assert int(oob) == (2 if n > 8 else 0)
    h = {k: a.double().cpu().numpy() for k, a in t.items()}
    ok = np.isfinite(h["x"]).all(1) & (h["x"] > 0).all(1)
    h = {k: a[ok] for k, a in h.items()}
    want_v, want_m = np.zeros((r1,) * dim + (dim,)), np.zeros((r1,) * dim)
    O.p2g(h["x"], h["v"], h["F"], h["C"], h["Jp"], h["mass"], h["mu0"], h["lam0"], O.ELASTIC, 1.0, float(res),
          1.0 / res, 1e-4, 1e-4, want_v, want_m)
    for got, want in ((gv, want_v), (gm, want_m)):
        error = np.abs(got.double().cpu().numpy() - want).max()
        assert error <= (1e-12 if dtype == torch.float64 else 130 * 6e-8) * np.abs(want).max()
