"""Chunk lists of more rows than one round of the chip, on both sides of each of
the rule's lines (rows in all, steps that single rows save, dense blocks): one
engine substep against the C oracle."""
import numpy as np
import pytest

from oracle import c_oracle as CO
from tests._parity import field_errors
from tests.gpu_helpers import engine_for, engine_roundtrip, oracle_copy_from, to_numpy_state, to_torch_state
from tests.test_chunk_sizes import _counts_state


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [
    [600] * 270,              # 810 rows, 1,080 steps as plain chunks: single
    [500] * 400 + [1],        # 801 rows and steps: plain
    [1153] * 160 + [700],     # 803 rows, most in dense blocks: grouped
    [300] * 1050 + [520],     # 2,103 rows: plain
    [1281] * 350 + [130],     # 2,101 rows in dense blocks: plain
], ids=["saves steps", "saves none", "dense", "many rows", "many dense rows"])
def test_substep_on_each_side(gpu, counts):
    st, pr = _counts_state(counts, 64, seed=len(counts))
    ts = to_torch_state(st, gpu)
    eng = engine_for(st, pr, gpu)
    out = engine_roundtrip(eng, ts, 1)
    eng.close()
    want = oracle_copy_from(ts, st)
    cs = CO.run(want, pr, 1, nthreads=8)
    n = len(want["x"])
    ref = {k: np.asarray(cs.arrays[k]).reshape(np.asarray(want[k]).shape) for k in ("x", "v", "F", "C", "Jp")}
    errs = field_errors(to_numpy_state(out), ref, pr["inv_dx"])
    # the per-substep bar of the engine's parity tests
    assert all(errs[k] <= 1e-5 for k in ("x", "v", "F")), (n, errs)
