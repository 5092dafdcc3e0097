"""Few activation rows on the split-K kernels' less common forms: rows too long for the LDS (sixteen waves a workgroup, some with one block
more than others), fewer rows than a group of eight (only those are copied), and several weights walked by rounds of tiles (nine rows and more).
Against the dot-product kernel of the staged path: the same block integers, f32 sums over a row's blocks in another order."""
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_fused_neighbours import qh  # noqa: F401

pytestmark = pytest.mark.gpu


def close(got, want, blocks):
    err = (got - want).double().norm(dim=1) / want.double().norm(dim=1)
    assert err.max().item() <= 4 * blocks * 2.0 ** -24 + 2e-7, err.max().item()


@pytest.mark.parametrize("dt,k", [("Q4K", 14336), ("Q5K", 11008), ("Q6K", 8448), ("Q4_0", 14400), ("Q8_0", 14336), ("Q4_0", 8512)])
@pytest.mark.parametrize("m,n", [(2, 16), (3, 1000), (5, 4096), (8, 257), (7, 4097), (9, 512)])
def test_long_rows(qh, dt, k, m, n):  # noqa: F811
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02, GgmlDType[dt]).weight
    x = torch.randn(m, k, generator=g, device="cuda")
    out = torch.full((m + 1, n), 7.0, device="cuda")
    qh.qmatmul(w, x, qh.FLAG_FORCE_SKINNY if n % 16 == 0 and k % 256 == 0 else 0, out=out[:m])
    assert bool((out[m] == 7.0).all())
    close(out[:m], qh.qmatmul(w, x, qh.FLAG_FORCE_MATVEC | qh.FLAG_STAGED_ACT), k // (32 if dt in ("Q8_0", "Q4_0") else 256))


@pytest.mark.parametrize("m,k,ns", [(9, 4096, (4096, 1024, 1024)), (16, 2304, (17, 40, 33)), (12, 2560, (4112, 8200)), (16, 4096, (16, 16400)),
                                    (9, 3840, (5000, 16, 16)), (10, 4352, (300, 200)), (16, 2048, (300, 200))])   # (the last two: past the rounds' ends)
def test_weights_by_rounds(qh, m, k, ns):  # noqa: F811
    g = torch.Generator(device="cuda").manual_seed(m + k)
    ws = [QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02, GgmlDType.Q4K).weight for n in ns]
    x = torch.randn(m, k, generator=g, device="cuda")
    for w, y in zip(ws, qh.qmatmul_multi(ws, x)):
        close(y, qh.qmatmul(w, x, qh.FLAG_FORCE_MATVEC | qh.FLAG_STAGED_ACT), k // 256)
