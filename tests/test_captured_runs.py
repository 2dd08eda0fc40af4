"""Runs and downloads in a graph of the caller's: every replay starts from the
memory that the captured run started from, whatever was downloaded in between."""
import pytest
import torch

from femflow_amd.engine import Engine, MaterialSpec, SceneSpec

pytestmark = pytest.mark.gpu
KEYS = ("x", "v", "F", "C", "Jp")


def _state(n, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    full = lambda a: torch.full((n,), a, device=dev)  # noqa: E731
    return dict(x=0.3 + 0.3 * torch.rand(n, 3, generator=g, device=dev),
                v=0.1 * torch.randn(n, 3, generator=g, device=dev), F=torch.eye(3, device=dev).repeat(n, 1, 1),
                C=torch.zeros(n, 3, 3, device=dev), Jp=full(1.0)), (full(1e-6), full(100.0), full(100.0))


@pytest.mark.parametrize("n", [50_000, (1 << 20) + 5])  # one and two passes of a download
@pytest.mark.parametrize("before", [(), (3,), (3, 3)])  # from an upload's records; from the tiles of either copy
def test_replays_equal_the_eager_run(gpu, n, before):
    """The captured run rebins at its start, so that each replay begins with the
    state before it; downloads in the graph and eager ones between the replays
    leave that state alone, and another upload replaces it where it was an upload
    or has its place (the first state copy)."""
    states = [_state(n, gpu, seed) for seed in (1, 2)]
    eng = Engine([SceneSpec(res=64, dt=1e-5, volume=1e-6)], [MaterialSpec("elastic")], n_max=n)
    eng.tune(use_graph=False)
    out, other = ({k: torch.empty_like(a) for k, a in states[0][0].items()} for _ in range(2))

    def upload(which):
        eng.upload(*states[which][0].values(), *states[which][1])

    def start():
        upload(0)
        for k in before:
            eng.run(k, check_oob=False)
            eng.request_rebin()

    def result():
        eng.run(6, check_oob=False)
        eng.download(*out.values())
        return {k: a.clone() for k, a in out.items()}

    with torch.cuda.stream(torch.cuda.Stream()):
        upload(1)
        wants = [result()]
        start()
        wants.insert(0, result())
        if len(before) == 1:  # its state is in the other copy, where no upload goes
            wants[1] = wants[0]
        start()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        graph.capture_begin()
        eng.run(6, check_oob=False)
        eng.download(*out.values())
        graph.capture_end()
        for replay in range(4):
            if replay == 3:
                upload(1)
            for a in out.values():
                a.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            for k in KEYS:
                assert torch.equal(out[k], wants[replay == 3][k]), (replay, k)
            if replay < 3:
                eng.download(*other.values())
                torch.cuda.synchronize()
                for k in KEYS:
                    assert torch.equal(other[k], wants[0][k]), (replay, k)
    del graph
    eng.close()
