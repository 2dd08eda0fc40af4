"""The reverse G2P's LDS arena holds 1,024 nodes: workgroups whose stencil box
is just inside and just outside of that (and of the smaller arena of the phase
P2G) against autograd through the FP64 reference."""
import numpy as np
import pytest
import torch

from oracle import mpm_torch as T
from tests.test_adjoint import _cube_scene, _rel


@pytest.mark.gpu
@pytest.mark.parametrize("length", [34, 35, 62, 63])  # boxes of 4 x 4 x (length + 2) nodes
def test_adjoint_step_of_a_strip(gpu, length):
    """256 particles, one workgroup, in arbitrary order in a strip of 2 x 2 x
    `length` cells, as particles in row-major cell order lie; half the bar of
    test_adjoint_step_matches_fp64_autograd."""
    from femflow_amd.adjoint import DenseStepper, RolloutConfig

    n, res, dt = 256, 72, 1e-4
    rng = np.random.default_rng(length)
    sc = _cube_scene(n, res, 11)
    u = rng.random((n, 3))
    u[0], u[1] = 0.01, 0.99  # both ends of the strip
    sc["x"] = (np.array([20, 30, 4]) + 0.5 + u * np.array([2, 2, length])) / res
    cfg = RolloutConfig(res=res, dt=dt, volume=sc["vol"], nsteps=1, hardening=1.2)
    st = DenseStepper(cfg, n, gpu)
    f32 = lambda a: torch.tensor(np.asarray(a), dtype=torch.float32, device=gpu).contiguous()  # noqa: E731
    x, v, F, C = f32(sc["x"]), f32(sc["v"]), f32(sc["F"]), f32(sc["C"])
    mass, mu0, lam0 = f32(sc["mass"]), f32(sc["mu0"]), f32(sc["lam0"])
    bars = [rng.standard_normal(s) for s in ((n, 3), (n, 3), (n, 3, 3), (n, 3, 3))]
    xb, vb, Fb, Cb = (f32(a) for a in bars)
    mub, lamb = torch.zeros_like(mu0), torch.zeros_like(lam0)
    st.adjoint(x, v, F, C, mass, mu0, lam0, xb, vb, Fb, Cb, mub, lamb)
    st.check_oob()
    ins = [t.detach().double().cpu().requires_grad_(True) for t in (x, v, F, C, mu0, lam0)]
    out = T.substep(*ins[:4], mass.double().cpu(), *ins[4:], res, dt, sc["vol"], hardening=1.2)
    ref = torch.autograd.grad(out, ins, grad_outputs=[f32(a).double().cpu() for a in bars])
    for name, g, r in zip("xvFCml", (xb, vb, Fb, Cb, mub, lamb), ref):
        assert _rel(g.cpu().numpy(), r.numpy()) < 1e-4, name
