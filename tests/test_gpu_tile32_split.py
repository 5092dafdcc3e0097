"""Q8_0 / Q4_0 prompts whose K is split inside the workgroup: up to 32 rows a wave by itself (one to eight column tiles a workgroup), beyond that
K halved between the waves (tiles of 32, 64 and 96 rows).  Rows of no whole tile, weight rows of no whole column tile, K steps that leave some
waves without one and a last step of fewer than eight blocks; against the dot-product kernel, which the oracle tests pin."""
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_fused_neighbours import qh  # noqa: F401
from tests.test_gpu_tile_tail import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("m,n,k", [(17, 4064, 4160), (32, 11997, 1088), (24, 16417, 576), (21, 32801, 1600)])   # 1, 2, 4, 8 column tiles
def test_few_rows(qh, dt, m, n, k):  # noqa: F811
    check(qh, dt, m, n, k)


@pytest.mark.parametrize("dt", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("m,n,k", [(33, 2080, 576), (64, 4100, 1088), (72, 2051, 320), (129, 131, 704), (300, 8160, 2048), (512, 4096, 2048),
                                   (77, 16250, 832), (190, 16250, 512)])   # (Q4_0: 96-row tiles, the second of two partly past the rows)
def test_k_halved(qh, dt, m, n, k):  # noqa: F811
    check(qh, dt, m, n, k)


@pytest.mark.parametrize("dt", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("m", [21, 77])
def test_rows_keep_apart(qh, dt, m):  # noqa: F811
    """Rows past the last one are garbage in the tiles, and a row of infinities and NaN stays by itself; nothing is written past y."""
    g = torch.Generator(device="cuda").manual_seed(m)
    w = QTensor.quantize(torch.randn(16250, 1088, generator=g, device="cuda") * 0.02, GgmlDType[dt]).weight
    x = torch.randn(m, 1088, generator=g, device="cuda")
    bad = x.clone()
    bad[3, 7], bad[3, 900] = float("inf"), float("nan")
    y, yb = qh.qmatmul(w, x), qh.qmatmul(w, bad)
    keep = [r for r in range(m) if r != 3]
    assert torch.equal(y[keep], yb[keep])
    out = torch.full((m + 1, 16250), 7.0, device="cuda")
    qh.qmatmul(w, x, out=out[:m])
    assert torch.equal(out[:m], y) and bool((out[m] == 7.0).all())
