"""Top-k selection at the edges of its histogram layouts."""
import pytest
import torch

from tread_amd import _hip

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n", [12287, 12288, 40960, 40961])
@pytest.mark.parametrize("clustered", [True, False])
def test_topk_select_on_both_histogram_layouts(n, clustered):
    g = torch.Generator().manual_seed(n)
    score = torch.randn(n, generator=g).abs() + 3 if clustered else torch.randn(n, generator=g) * 100
    score = score.to(torch.bfloat16)
    k = n // 5
    order = sorted(range(n), key=lambda i: (-score[i].item(), i))[:k]  # ties to the lowest index
    assert _hip.topk_select(score.to(DEV), k).cpu().tolist() == sorted(order)
