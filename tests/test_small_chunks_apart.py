"""Small chunks of engines with many scenes on both sides of the number from
which they go to a launch of their own."""
import pytest
import torch

from tests.test_small_chunks import KEYS, _run, _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra", [761, 762, 900])  # 767, 768 and 906 small chunks in all
@pytest.mark.parametrize("splits", [(1,), (2, 3)])
def test_results_do_not_depend_on_the_launch(gpu, extra, splits):
    """Scenes of one block each: those at the edges of a row, of a wave's two and
    of the limit of 128, and `extra` of 3 particles; against engines of one
    scene (the bars of test_small_chunks), and the same from run to run."""
    counts = (1, 63, 64, 65, 127, 128, 129, 513) + (3,) * extra
    s = _state(counts, gpu)
    outs = [_run(s, s["scene"], len(counts), splits) for _ in range(2)]
    for k in KEYS:
        assert torch.equal(outs[0][k], outs[1][k]), k
    for i in (0, 1, 2, 3, 4, 5, 6, 8, len(counts) - 1):
        at = torch.nonzero(s["scene"] == i).flatten()
        alone = _run({k: a[at].contiguous() for k, a in s.items()}, None, 1, splits)
        for k in KEYS:
            a, b = outs[0][k][at], alone[k]
            assert float((a - b).abs().max()) <= (1e-5 if k == "C" else 1e-6) * float(b.abs().max()), (i, k)
