"""Two to four activation rows on either side of the weight row counts where the one-launch kernel hands over to the quantizer
and the split-K kernel: against the dot-product kernel of the staged path, which the oracle tests pin (the same block integers,
f32 sums over a row's blocks in another order: 2^-24 an addition and two products of each block)."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from candle_amd.quantized import GgmlDType, QTensor  # noqa: E402
from tests.test_gpu_fused_neighbours import qh  # noqa: E402,F401


@pytest.mark.parametrize("dt,m,n,k", [("Q4K", 2, 6786, 512), ("Q5K", 2, 15258, 1024), ("Q4K", 2, 7680, 1280), ("Q6K", 3, 5566, 768),
                                      ("Q5K", 3, 5055, 1536), ("Q4K", 3, 14329, 2048), ("Q6K", 4, 6378, 1024), ("Q6K", 3, 20875, 3072),
                                      ("Q4K", 4, 17, 1280), ("Q4_0", 3, 16405, 512), ("Q4_0", 4, 16150, 1024), ("Q3K", 4, 4334, 512),
                                      ("Q2K", 4, 4334, 512)])
def test_either_side_of_the_hand_over(qh, dt, m, n, k):  # noqa: F811
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    dense = torch.randn(n, k, generator=g, device="cuda") * 0.02
    x = torch.randn(m, k, generator=g, device="cuda")
    for rows in (n - 1, n):
        w = QTensor.quantize(dense[:rows].contiguous(), GgmlDType[dt]).weight
        got, want = qh.qmatmul(w, x), qh.qmatmul(w, x, qh.FLAG_FORCE_MATVEC | qh.FLAG_STAGED_ACT)
        err = (got - want).double().norm(dim=1) / want.double().norm(dim=1)
        blocks = k // (32 if dt == "Q4_0" else 256)
        assert err.max().item() <= 4 * blocks * 2.0 ** -24 + 2e-7, (rows, err.max().item())
