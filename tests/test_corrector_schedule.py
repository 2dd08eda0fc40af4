"""The corrector turned on between two runs: its substeps use the chunk list
that it needs, whatever the engine ran before."""
import pytest
import torch

from tests.test_cadence import _download, _engine, _state, _upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("before", [1, 5])
def test_enabling_the_corrector_rebuilds_the_chunks(gpu, before):
    """Equal, to the last bit, to the same calls with a rebin asked for at the
    switch (a calm scene: no particle leaves its chunk's arena, so that nothing
    adds in an order of its own)."""
    from femflow_amd.corrector import CorrectorMLP

    zero = torch.zeros_like(CorrectorMLP(device=gpu).params)
    s = _state(gpu, 0.005)
    outs = []
    for rebin in (False, True):
        eng = _engine(48)
        eng.set_corrector(zero, 1e-6, 1.0, enable=False)
        _upload(eng, s)
        eng.run(before)
        eng.set_corrector(zero, 1e-6, 1.0, enable=True)
        if rebin:
            eng.request_rebin()
        eng.run(3)
        eng.run(2)
        outs.append(_download(eng, s))
        eng.close()
    for k in outs[0]:
        assert torch.equal(outs[0][k], outs[1][k]), k


def test_disabling_and_enabling_again(gpu):
    """A network of zeros corrects nothing: plain substeps between corrected
    ones, on the same chunk list, leave the bits alone."""
    from femflow_amd.corrector import CorrectorMLP

    zero = torch.zeros_like(CorrectorMLP(device=gpu).params)
    s = _state(gpu, 0.005)
    outs = []
    for toggles in (False, True):
        eng = _engine(48)
        eng.set_corrector(zero, 1e-6, 1.0, enable=True)
        _upload(eng, s)
        for k in (2, 1, 2):
            if toggles and k == 1:
                eng.set_corrector(None, enable=False)
            eng.run(k)
            if toggles and k == 1:
                eng.set_corrector(zero, 1e-6, 1.0, enable=True)
        outs.append(_download(eng, s))
        eng.close()
    for k in outs[0]:
        assert torch.equal(outs[0][k], outs[1][k]), k
