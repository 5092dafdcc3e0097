"""The offset terms of Q4_1 / Q5_1 / Q2K behind the dot-product kernels, where a row's bits may not depend on how many rows a call has."""
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_fused_neighbours import qh  # noqa: F401

pytestmark = pytest.mark.gpu


def weight_and_rows(dt, n, k, m):
    g = torch.Generator(device="cuda").manual_seed(n + k)
    w = QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02 + 0.01, GgmlDType[dt]).weight
    return w, torch.randn(m, k, generator=g, device="cuda")


@pytest.mark.parametrize("dt,k", [("Q4_1", 64), ("Q2K", 256)])
def test_more_rows_than_a_grid_has_groups(qh, dt, k):  # noqa: F811
    """Groups of four rows in a grid's second dimension: 65535 of them are 262140 rows.  The rows repeat every 1000, and so do the results."""
    m = 4 * 65535 + 7
    w, few = weight_and_rows(dt, 3, k, 1000)
    y = qh.qmatmul(w, few[torch.arange(m, device="cuda") % 1000])
    want = qh.qmatmul(w, few)
    assert torch.equal(y, want[torch.arange(m, device="cuda") % 1000])
