"""Particles deferred to FP64 are finished inside the grid update (plain runs,
recorded states and frames) or by a launch of their own ahead of it (engines with
the corrector, whose features are summed from finished particles)."""
import numpy as np
import pytest
import torch

from oracle import mpm_oracle as O
from tests.gpu_helpers import engine_for, engine_roundtrip, to_torch_state
from tests.test_engine_edges import _rotation

pytestmark = pytest.mark.gpu


def test_deferred_launch_matches_the_grid_update(gpu):
    """A corrector of zeros corrects nothing, so both kinds of engine take the
    same substeps; the scene and the bars are those of
    test_engine_deferred_in_grid_update_matches_separate_pass."""
    from femflow_amd.corrector import CorrectorMLP

    rng = np.random.default_rng(13)
    st, pr = O.scene_3d_cubes(n=20000, res=32, seed=14, side=0.25, corners=((0.3, 0.35, 0.3),),
                              materials=(O.MATERIALS_C2[0],), vel_sigma=0.2)
    n, k = len(st["x"]), 4
    F = st["F"].reshape(n, 3, 3)
    for p in rng.choice(n, size=600, replace=False):
        F[p] = _rotation(rng) @ np.diag([1.02, 0.98, 2e-4]) @ _rotation(rng)
    st["F"] = F.reshape(st["F"].shape)
    ts = to_torch_state(st, gpu)
    plain = engine_for(st, pr, gpu, sort_every=48)
    in_grid = engine_roundtrip(plain, ts, k)
    fb_grid = plain.fallback_count()
    plain.close()
    net = engine_for(st, pr, gpu, sort_every=48)
    net.set_corrector(torch.zeros_like(CorrectorMLP(device=gpu).params), float(ts["mass"].mean()), 1.0)
    apart = engine_roundtrip(net, ts, k)
    fb_apart = net.fallback_count()
    net.close()
    assert min(fb_grid, fb_apart) >= 4 * 500 and abs(fb_grid - fb_apart) <= 0.01 * fb_apart, (fb_grid, fb_apart)
    bars = {"x": 1e-5, "v": 1e-5, "F": 1e-5, "C": 1e-4, "Jp": 1e-5}
    for f, bar in bars.items():
        scale = float(apart[f].abs().max()) + 1e-30
        assert float((in_grid[f] - apart[f]).abs().max()) < bar * scale, f
