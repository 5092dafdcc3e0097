"""Q4_0 prompts of 65 to 96 rows in one row of 96-row tiles: the instance that leaves out the upper sixteen rows of the last 32 where they are padding,
and its neighbour.  Against the dot-product kernel of the staged path: the same block integers, f32 sums over a row's blocks in another order."""
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_fused_neighbours import qh  # noqa: F401
from tests.test_gpu_few_rows_long import close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [65, 77, 80, 81])
@pytest.mark.parametrize("n,k", [(32000, 512), (31999, 576), (28001, 1280), (24003, 1088)])   # (the last: steps of no whole length)
def test_padding_rows(qh, m, n, k):  # noqa: F811
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02, GgmlDType.Q4_0).weight
    x = torch.randn(m, k, generator=g, device="cuda")
    x[m - 1, 5] = 40.0
    out = torch.full((m + 1, n), 7.0, device="cuda")
    qh.qmatmul(w, x, out=out[:m])
    assert bool((out[m] == 7.0).all())
    close(out[:m], qh.qmatmul(w, x, qh.FLAG_FORCE_MATVEC | qh.FLAG_STAGED_ACT), k // 32)
