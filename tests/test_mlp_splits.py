"""Row counts at which the weight gradients' launch has as many splits as its
scratch memory has room for (56)."""
import ctypes as ct

import numpy as np
import pytest
import torch

from oracle import mlp_oracle as M
from tests.test_corrector import _data, _params


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [56 * 384 - 17, 56 * 384, 56 * 256 - 127])
def test_gradients_with_every_split(gpu, rows):
    """21,487 rows: 56 splits of 384, the last one short; 21,504: all full;
    14,209: 56 of 256.  Against the NumPy restatement and the form without scratch
    memory, to the bars of test_mlp_gradients_at_row_edges."""
    from femflow_amd import _lib
    from femflow_amd.corrector import CorrectorMLP, to_bf16_features

    X, T, w = _data(rows, rows)
    p = _params(6)
    net = CorrectorMLP(device=gpu, params=torch.from_numpy(p))
    Xg = to_bf16_features(X, gpu)
    net.loss_grads(Xg, torch.tensor(T, dtype=torch.float32), torch.tensor(w, dtype=torch.float32))
    _, gref, _ = M.loss_and_grads(p.astype(np.float64), X, T, w)
    assert np.linalg.norm(net.grads.double().cpu().numpy() - gref) <= 1e-3 * np.linalg.norm(gref)
    b = ct.c_int64()
    _lib.check(_lib.load().mpm_mlp_backward_workspace_bytes(rows, ct.byref(b)))
    assert b.value == 4 * p.size * 56
    atomic = torch.zeros_like(net.grads)
    _lib.check(_lib.load().mpm_mlp_backward(
        torch.cuda.current_stream().cuda_stream, net.packed.data_ptr(), Xg.data_ptr(), rows, net.H1.data_ptr(),
        net.H2.data_ptr(), net.dY.data_ptr(), net.dH2.data_ptr(), net.dH1.data_ptr(), atomic.data_ptr()))
    assert float((atomic - net.grads).norm()) <= 1e-5 * float(net.grads.norm())
