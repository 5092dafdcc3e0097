"""Q8_0 / Q4_0 prompts whose K is split inside the workgroup: up to 32 rows a wave by itself (one to eight column tiles a workgroup), beyond that
K halved between the waves (tiles of 32, 64 and 96 rows).  Rows of no whole tile, weight rows of no whole column tile, K steps that leave some
waves without one and a last step of fewer than eight blocks; against the dot-product kernel, which the oracle tests pin."""
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_few_rows_long import close
from tests.test_gpu_fused_neighbours import qh  # noqa: F401
from tests.test_gpu_tile_tail import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("m,n,k", [(17, 4064, 4160), (32, 11997, 1088), (24, 16417, 576), (21, 32801, 1600)])   # 1, 2, 4, 8 column tiles
def test_few_rows(qh, dt, m, n, k):  # noqa: F811
    check(qh, dt, m, n, k)


@pytest.mark.parametrize("dt", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("m,n,k", [(33, 2080, 576), (64, 4100, 1088), (72, 2051, 320), (129, 131, 704), (300, 8160, 2048), (512, 4096, 2048),
                                   (77, 16250, 832), (190, 16250, 512)])   # (the last, Q4_0: 96-row tiles, the second of two partly past the rows)
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


@pytest.mark.parametrize("dt", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("m,n,k", [(17, 130, 1536), (32, 130, 1088), (24, 1000, 768), (24, 1000, 576), (20, 1000, 512), (20, 1000, 320), (17, 33788, 1536),
                                   (17, 33788, 1088),                                                                    # 1, 2, 4, 8 column tiles
                                   (32, 4096, 12288), (32, 4090, 12224), (17, 8192, 9984), (17, 8190, 9792), (19, 13996, 6144), (19, 13996, 6208),
                                   (31, 26366, 3072), (31, 26366, 3136), (25, 51106, 1600), (25, 52343, 1536),           # ... of 40 MB and more
                                   (33, 130, 512), (33, 130, 320), (48, 16470, 1536), (48, 16470, 3136), (129, 13996, 512), (129, 13996, 320),
                                   (65, 22655, 512), (65, 22655, 320),                                                   # K halved: 32, 64, 96 rows
                                   (33, 130, 1024), (33, 130, 832), (17, 65950, 1536), (17, 65950, 1600), (33, 33788, 256), (33, 33788, 320),
                                   (65, 43684, 256), (65, 43684, 320)])                                                  # K over workgroups or not at all
def test_each_form(qh, dt, m, n, k):  # noqa: F811
    """Every tile launch of these types by whole steps of K and not, and once more on the rows left in the workspace, where no quantizer
    launch clears the output of the forms that add to it."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02, GgmlDType[dt]).weight
    x = torch.randn(m, k, generator=g, device="cuda")
    ws = qh.Workspace()
    want = qh.qmatmul(w, x, qh.FLAG_FORCE_MATVEC | qh.FLAG_STAGED_ACT)
    close(qh.qmatmul(w, x, qh.FLAG_FORCE_GEMM, workspace=ws), want, k // 32)
    out = torch.full((m + 1, n), 7.0, device="cuda")
    qh.qmatmul(w, x, qh.FLAG_FORCE_GEMM | qh.FLAG_REUSE_ACT, out=out[:m], workspace=ws)
    close(out[:m], want, k // 32)
    assert bool((out[m] == 7.0).all())
