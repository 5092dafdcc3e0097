"""More than 16 rows of small K-quant weights in groups of 16 or 32 rows beside each other: rows of no whole group, weight rows of no whole tile,
fewer blocks than waves and some waves with one more than others.  Against the dot-product kernel of the staged path: the same block integers,
f32 sums over a row's blocks in another order."""
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_fused_neighbours import qh  # noqa: F401
from tests.test_gpu_few_rows_long import close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["Q4K", "Q5K", "Q6K", "Q3K", "Q2K", "Q8_0", "Q4_0", "Q4_1", "Q5_1"])
@pytest.mark.parametrize("m,n,k", [(17, 16, 2304), (31, 2048, 2560), (33, 33, 256), (40, 1000, 2304), (48, 130, 13312), (64, 384, 512), (100, 411, 3584),
                                   (257, 40, 256), (500, 256, 1024), (96, 2047, 1792), (128, 1024, 4096), (1025, 24, 768)])
def test_groups(qh, dt, m, n, k):  # noqa: F811
    run(qh, dt, m, n, k)


def run(qh, dt, m, n, k):  # noqa: F811
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02, GgmlDType[dt]).weight
    x = torch.randn(m, k, generator=g, device="cuda")
    out = torch.full((m + 1, n), 7.0, device="cuda")
    qh.qmatmul(w, x, out=out[:m])
    assert bool((out[m] == 7.0).all())
    close(out[:m], qh.qmatmul(w, x, qh.FLAG_FORCE_MATVEC | qh.FLAG_STAGED_ACT), k // (256 if dt.endswith("K") else 32))
    bad = x.clone()
    bad[m // 2, 3], bad[m // 2, k - 1] = float("inf"), float("nan")
    keep = [r for r in range(m) if r != m // 2]
    # (shapes whose choice is the tile kernel: without parts added up atomically)
    assert torch.equal(qh.qmatmul(w, bad, qh.FLAG_DETERMINISTIC)[keep], qh.qmatmul(w, x, qh.FLAG_DETERMINISTIC)[keep])


@pytest.mark.parametrize("dt", ["Q8_0", "Q4_0", "Q5_0", "Q4_1"])
@pytest.mark.parametrize("m,n,k", [(17, 16, 320), (20, 2050, 2112), (33, 100, 4160), (129, 31, 576), (40, 1500, 960)])
def test_steps_of_no_whole_length(qh, dt, m, n, k):  # noqa: F811
    run(qh, dt, m, n, k)


@pytest.mark.parametrize("dt", ["Q4K", "Q5K", "Q6K", "Q3K", "Q2K", "Q8_0", "Q4_0", "Q4_1", "Q5_1"])
@pytest.mark.parametrize("m,n,k", [(17, 4090, 2304), (24, 2065, 2560), (25, 4096, 2304), (32, 3000, 2816), (20, 3001, 512), (32, 4000, 1024), (24, 4100, 2304),
                                   (31, 4130, 768), (12, 1000, 2304), (16, 4100, 3840)])
def test_all_rows_in_one_workgroup(qh, dt, m, n, k):  # noqa: F811
    """Nine to 32 rows, from 17 on of too many weight rows for groups: two to four groups of eight, resident (up to 4096 weight rows), by rounds
    of tiles and not."""
    run(qh, dt, m, n, k)
