"""2D G2P gather (femflow/solvers/mpm/two_d/g2p.py:5-47) on the GPU."""
from __future__ import annotations

from .... import _lib
from .. import _phase


def g2p(inv_dx, dt, grid_velocity, x, v, F, C, Jp, model: str = "neo_hookean"):
    """Gather, advect, update F; the SVD rebuild and Jp update run for every
    particle, the singular value clamp only for ``model == "snow"``."""
    res = int(grid_velocity.shape[0]) - 1
    sp = _phase.StagedParticles(x, v, F, C, Jp, None, None, None)
    prm = _phase.make_params(2, res, inv_dx, 1.0 / inv_dx, dt, check_oob=False)
    _lib.require_gpu()
    _phase.launch_g2p(sp, prm, sp.struct(), _phase.g2p_kind(model), grid_velocity)
    sp.commit()
