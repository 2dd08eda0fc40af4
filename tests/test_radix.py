"""The stable sort behind the binning at the edges of its plan: tiles of 1,024,
2,048 and 4,096 keys and their remainders, one, two and three passes over
digits of 8 to 11 bits, all keys equal."""
import numpy as np
import pytest
import torch

from oracle import mpm_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,res,dim,layout,spread", [
    (1, 16, 3, "blocked", 1.0),
    (1023, 3, 2, "rowmajor", 1.0),            # 16 keys, one pass
    (1025, 40, 2, "blocked", 1.0),            # 11 bits, one pass
    (70_001, 16, 3, "blocked", 0.0),          # all equal
    (65_536, 60, 3, "blocked", 0.9),          # two passes of 9 bits
    (1 << 19, 128, 3, "blocked", 0.5),        # the last of the smallest tiles
    ((1 << 19) + 1, 96, 3, "rowmajor", 0.7),  # the first of the middle ones
    (1 << 20, 128, 3, "rowmajor", 0.3),
    ((1 << 20) + 77, 1000, 3, "rowmajor", 1.0),  # largest tiles, three passes
])
def test_binning_is_the_stable_order(gpu, n, res, dim, layout, spread):
    from femflow_amd.engine import bin_particles

    x = (0.5 + spread * (np.random.default_rng(n).random((n, dim)) - 0.5)).astype(np.float32)
    ref = O.bin_keys(x, float(res), res, layout=layout)
    xt = torch.tensor(x, device=gpu)
    for _ in range(2):  # a second call meets the first one's scratch memory
        keys, perm = bin_particles(xt, res, float(res), layout)
        assert np.array_equal(keys.cpu().numpy().view(np.uint32), ref)
        assert np.array_equal(perm.cpu().numpy().view(np.uint32), np.argsort(ref, kind="stable"))
