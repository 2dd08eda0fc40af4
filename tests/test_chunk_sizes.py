"""Blocks whose particle counts sit at the edges of the chunk list's rules
(one row, just over one, a pair less than 3/4 full, many rows; few and many
rows in all; one scene and many): one engine substep against the FP64 oracle."""
import numpy as np
import pytest
import torch

from oracle import mpm_oracle as O
from tests._parity import field_errors
from tests.gpu_helpers import engine_for, engine_roundtrip, oracle_copy_from, to_numpy_state, to_torch_state


def _counts_state(counts, res, seed):
    """counts[i] particles at random in the i-th 4x4x4-cell block of a row of
    blocks away from the walls."""
    rng = np.random.default_rng(seed)
    x = []
    per_row = res // 4 - 4
    for i, c in enumerate(counts):
        b = np.array([2 + i // (per_row * per_row), 2 + (i // per_row) % per_row, 2 + i % per_row])
        x.append((4 * b + 0.5 + 4 * rng.random((c, 3))) / res)
    st, pr = O.scene_3d_cubes(n=sum(counts), res=res, seed=seed)
    st["x"] = np.concatenate(x)
    n = len(st["x"])
    B = 30.0 * rng.normal(size=(3, 3))
    st["v"] = (st["x"] - 0.5) @ B.T
    st["C"] = np.broadcast_to(B, (n, 3, 3)).copy()
    st["F"] = np.eye(3) + 0.004 * rng.normal(size=(n, 3, 3))
    return st, pr


@pytest.mark.gpu
@pytest.mark.parametrize("counts,res", [
    ([1, 255, 256, 257, 383, 384, 385, 511, 512, 513, 667, 768, 769, 1025], 64),  # few rows in all
    ([1333] * 70 + [260, 1153, 5], 64),                                          # most rows dense: grouped
    ([600] * 160 + [3000], 64),                                                  # many rows, not dense: single
])
def test_substep_at_chunk_edges(gpu, counts, res):
    st, pr = _counts_state(counts, res, seed=len(counts))
    ts = to_torch_state(st, gpu)
    eng = engine_for(st, pr, gpu)
    out = engine_roundtrip(eng, ts, 1)
    eng.close()
    want = oracle_copy_from(ts, st)
    O.substep(want, pr)
    # the per-substep bar of the engine's parity tests
    errs = field_errors(to_numpy_state(out), want, pr["inv_dx"])
    assert all(errs[k] <= 1e-5 for k in ("x", "v", "F")), errs
