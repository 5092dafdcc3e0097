"""The offset terms of Q4_1 / Q5_1 / Q2K behind the dot-product kernels, where a row's bits may not depend on how many rows a call has."""
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from oracle import cpu_oracle as orc
from tests.test_gpu_few_rows_long import close
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


@pytest.mark.parametrize("dt", ["Q4_1", "Q5_1", "Q2K"])
@pytest.mark.parametrize("n,k", [(8, 256), (15, 4352), (100, 2560), (1000, 2816), (4100, 512), (4100, 2304)])
def test_bits_do_not_depend_on_the_rows_beside(qh, dt, n, k):  # noqa: F811
    """Across the lines between the kernels (four rows, 64 rows, a count of outputs), with rows and weight rows of no whole tile."""
    flags = qh.FLAG_FORCE_MATVEC | qh.FLAG_STAGED_ACT
    w, x = weight_and_rows(dt, n, k, 200)
    y = qh.qmatmul(w, x, flags)
    for m in (1, 4, 5, 7, 20, 21, 33, 64, 65):
        assert torch.equal(qh.qmatmul(w, x[:m].contiguous(), flags), y[:m]), m


@pytest.mark.parametrize("dt", ["Q4_1", "Q5_1", "Q2K"])
@pytest.mark.parametrize("n,k,m", [(15, 256, 6), (33, 2816, 31), (70, 4352, 65), (5, 2560, 66)])
def test_against_the_oracle(qh, dt, n, k, m):  # noqa: F811
    w, x = weight_and_rows(dt, n, k, m)
    want = orc.matmul(getattr(orc, dt), x.cpu().numpy(), w.to_ggml(), n)
    close(qh.qmatmul(w, x, qh.FLAG_FORCE_MATVEC | qh.FLAG_STAGED_ACT).cpu(), torch.from_numpy(want), k // (256 if dt == "Q2K" else 32))
