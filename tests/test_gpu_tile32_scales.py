"""Block scales at the ends of f16 in the tile kernels of Q8_0 and Q4_0, where the product of two scales comes from the matrix cores: weights and
activations whose scales are subnormal, or large, beside ordinary ones.  Against the dot-product kernel of the staged path: the same block integers
and scales, f32 sums over a row's blocks in another order."""
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_few_rows_long import close
from tests.test_gpu_fused_neighbours import qh  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("m,n,k", [(24, 8200, 1088), (77, 28001, 1280), (200, 2080, 576), (300, 9000, 512)])   # few rows, K halved, tiles
@pytest.mark.parametrize("w_scale,x_scale", [(1e-5, 1.0), (1.0, 2e-5), (3e-5, 1e-5), (3e4, 2e4)])
def test_scales_at_the_ends(qh, dt, m, n, k, w_scale, x_scale):  # noqa: F811
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = torch.randn(n, k, generator=g, device="cuda") * w_scale
    w[::3] *= 0.02
    x = torch.randn(m, k, generator=g, device="cuda") * x_scale
    x[::2, : k // 2] *= 30.0
    w = QTensor.quantize(w, GgmlDType[dt]).weight
    ref = qh.qmatmul(w, x, qh.FLAG_FORCE_MATVEC | qh.FLAG_STAGED_ACT)
    assert bool((ref != 0).any())
    close(qh.qmatmul(w, x), ref, k // 32)
