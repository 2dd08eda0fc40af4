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


@pytest.mark.parametrize("short", [(5,), (5, 2), (8, 8, 1)])
def test_counts_outlast_runs_too_short_to_use_them(gpu, short):
    """Unchecked runs of at most 8 substeps after an upload cannot use its
    counts; the first longer one then uses those of the run before it, and
    rebins as it would have right after the upload: 8 substeps (from the order
    of the short runs), then by the fast particles' cadence of 8."""
    fast = _state(gpu, 0.2)
    eng = _engine(48)
    _upload(eng, fast)
    for k in short:
        eng.run(k, check_oob=False)
    assert _segments(eng, 48) == 1 + 5
    eng.close()


def test_recorded_sums_leave_the_counts(gpu):
    """A run that records sums keeps its schedule in one piece; the next one
    follows the speeds."""
    fast = _state(gpu, 0.2)
    eng = _engine(48)
    _upload(eng, fast)
    eng.run(12, sums=torch.empty(12, 8, dtype=torch.float64, device=gpu), check_oob=False)
    assert _segments(eng, 48) == 1 + 5
    eng.close()


@pytest.mark.parametrize("after_run", [False, True])
def test_a_sample_leaves_the_counts(gpu, after_run):
    """One P2G and grid update between an upload (or a checked run) and a run
    leaves the counts that the run reads: the fast particles' cadence of 8 from
    the sample's order on."""
    from femflow_amd.corrector import CorrectorMLP

    fast = _state(gpu, 0.2)
    eng = _engine(48)
    eng.set_corrector(torch.zeros_like(CorrectorMLP(device=gpu).params), 1e-6, 1.0, enable=False)
    _upload(eng, fast)
    if after_run:
        eng.run(4)
    eng.p2g_grid_only()
    assert _segments(eng, 48) == 6
    eng.close()


@pytest.mark.parametrize("split", [False, True])
def test_a_cadence_ends_without_new_counts(gpu, split):
    """Moving particles, counted after the upload only: the cadence K that the
    counts give holds for the 8 substeps while they are read and 192 more, up to
    the rebin after them, in one call or two; then sort_every."""
    s = _state(gpu, 0.05)
    eng = _engine(48)
    _upload(eng, s)
    per48 = _segments(eng, 48)
    assert 2 <= per48 <= 4  # 24, 16 or 12
    K = 48 // per48
    held = -(-200 // K)  # segments
    _upload(eng, s)
    eng.kernel_timing(True)
    for k in (held * K, 480 - held * K) if split else (480,):
        eng.run(k, check_oob=False)
    got = eng.kernel_times()["p2g"][1]
    eng.kernel_timing(False)
    assert got == held - (-(480 - held * K) // 48)
    assert eng.oob_count() == 0
    eng.close()
