"""The speed counts behind the engine's rebin cadence: which run they reach,
and how long a run waits for them."""
import time

import pytest
import torch

from tests.test_cadence import _engine, _segments, _state, _upload

pytestmark = pytest.mark.gpu


def _spin(seconds):
    """Hold back the current stream for about this long."""
    e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    torch.cuda._sleep(1000)
    e[0].record()
    torch.cuda._sleep(10_000_000)
    e[1].record()
    torch.cuda.synchronize()
    torch.cuda._sleep(int(10_000_000 * 1e3 * seconds / e[0].elapsed_time(e[1])))


@pytest.mark.parametrize("first,second,segments", [(0.2, 0.005, 1), (0.005, 0.2, 1)])
def test_late_counts_reach_no_other_run(gpu, first, second, segments):
    """A stream that holds back a run for longer than the run waits: the call
    returns, and the counts that it sends later are not taken for those of the
    run after it, which keeps sort_every."""
    states = [_state(gpu, s) for s in (first, second)]
    eng = _engine(48)
    _upload(eng, states[0])
    eng.run(1)
    with torch.cuda.stream(torch.cuda.Stream()):
        _spin(1.0)
        _upload(eng, states[0])
        start = time.monotonic()
        eng.run(48, check_oob=False)
        assert time.monotonic() - start < 0.7  # 0.2 s, and the launches
        _upload(eng, states[1])
        assert _segments(eng, 48) == segments
        # counts that have arrived in the meantime do not stop later probes
        _upload(eng, states[0])
        assert _segments(eng, 48) == (6 if first > 0.1 else 1)
    eng.close()
