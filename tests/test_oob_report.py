"""What the engine's counter of off-grid stencils is reported as: an exhausted
wait of the grid update (2^40 and more) is not a number of particles, whichever
call finds it.  The counter is stubbed; no GPU."""
import pytest
import torch

from femflow_amd.engine import Engine, SceneSpec


class _Lib:
    """Every entry point succeeds; the counter reads as given."""

    def __init__(self, count):
        self.count = count

    def __getattr__(self, name):
        def call(*args):
            if name == "mpm_ctx_oob_count":
                args[1]._obj.value = self.count
            return 0

        return call


def _engine(count):
    eng = Engine.__new__(Engine)
    eng._L, eng._h, eng.n, eng.scenes = _Lib(count), None, 2, [SceneSpec(res=4, dt=1e-4)]
    eng._sync_stream = lambda: None
    eng._check_tensor = lambda *a, **k: None
    return eng


def _calls():
    z = lambda *s: torch.zeros(s)  # noqa: E731
    state = (z(3, 2, 3), z(3, 2, 3), z(3, 2, 3, 3), z(3, 2, 3, 3), z(3, 2))
    return {
        "run": lambda e: e.run(3),
        "run_states": lambda e: e.run_states(3, *state),
        "run_states_grids": lambda e: e.run_states(3, *state, grids=z(3, 7 * 125)),
        "run_frames": lambda e: e.run_frames(3, z(3, 2, 3)),
    }


@pytest.mark.parametrize("call", ["run", "run_states", "run_states_grids", "run_frames"])
@pytest.mark.parametrize("count,message", [
    (0, None), (1, "1 particle stencil"), ((1 << 40) - 1, "particle stencil"), (1 << 40, "did not finish in time"),
    ((1 << 40) + 5, "did not finish in time")])
def test_counter_reports(call, count, message):
    eng, run = _engine(count), _calls()[call]
    if message is None:
        run(eng)
        return
    with pytest.raises(RuntimeError, match=message):
        run(eng)
