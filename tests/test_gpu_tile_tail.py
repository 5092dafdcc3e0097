"""Prompts whose 128-row tiles leave a last round of workgroups at most half full: that round's tiles are 64 or 32 rows high.
Against the dot-product kernel, which the oracle tests pin: the same block integers, f32 sums over the blocks of a row and the
f16 min term apart, an addition of either per block: 2^-24 each, and as many again for the two products of a block."""
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_fused_neighbours import qh  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["Q4K", "Q5K", "Q6K", "Q8_0", "Q4_0"])
@pytest.mark.parametrize("m,n,k", [(1100, 8192, 512),          # 288 tiles: 32 left, as 32-row tiles, some past the last row
                                   (1025, 8192 - 17, 256),     # ragged weight rows, one live row in the last strip
                                   (1000, 11264, 512),         # 352 tiles: 96 left, as 64-row tiles
                                   (1024, 12288, 256),         # 384: 128 left, the most that 64-row tiles take
                                   (1024, 8448, 256),          # 264: 8 left
                                   (1024, 12544, 256)])        # 392: too many left
def test_last_round_in_shorter_tiles(qh, dt, m, n, k):  # noqa: F811
    check(qh, dt, m, n, k)


@pytest.mark.parametrize("dt", ["Q4K", "Q6K", "Q8_0"])
@pytest.mark.parametrize("m,n,k", [(2100, 6400, 256),          # 17 x 25 tiles in strips of eight columns: the last strip has one
                                   (17000, 700, 256),          # three columns only
                                   (4400, 1800, 512)])         # one whole strip
def test_several_rounds_in_strips(qh, dt, m, n, k):  # noqa: F811
    check(qh, dt, m, n, k)


@pytest.mark.parametrize("dt", ["Q4K", "Q5K", "Q6K", "Q8_0", "Q4_0"])
@pytest.mark.parametrize("m,n,k", [(511, 2048, 512), (512, 2048, 512), (2000, 524, 512), (2001, 525, 512), (2200, 480, 4096)])
def test_results_around_the_size_of_streamed_ones(qh, dt, m, n, k):  # noqa: F811
    """2^20 results and more are stored non-temporal: whole and halved K, ragged columns, on both sides of the line."""
    check(qh, dt, m, n, k)


@pytest.mark.parametrize("dt", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("m,n,k", [(1100, 8192, 320), (1000, 11264 - 3, 576)])
def test_rows_of_no_whole_step(qh, dt, m, n, k):  # noqa: F811
    check(qh, dt, m, n, k)


@pytest.mark.parametrize("dt", ["Q4K", "Q5K", "Q6K", "Q8_0", "Q4_0"])
@pytest.mark.parametrize("m,n,k", [(1100, 8192, 512), (1025, 8160, 256), (1000, 11264, 512), (512, 4096, 1024)])   # (the last: 64 rows, K halved)
def test_integers_of_both_heights(qh, dt, m, n, k):  # noqa: F811
    """The same launches storing their block integers (the min term's as well): every one equals the dot-product kernels'."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02, GgmlDType[dt]).weight
    x = torch.randn(m, k, generator=g, device="cuda")
    got, mins = qh.qmatmul_int_dots_mfma(w, x, qh.MFMA_TILE | qh.MFMA_INT_MIN)
    want, want_mins = qh.qmatmul_int_dots(w, x)
    assert torch.equal(got, want)
    assert mins is None or torch.equal(mins.to(torch.int32), want_mins)


def check(qh, dt, m, n, k):  # noqa: F811
    block = 32 if dt in ("Q8_0", "Q4_0") else 256
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02, GgmlDType[dt]).weight
    x = torch.randn(m, k, generator=g, device="cuda")
    got = qh.qmatmul(w, x)
    want = qh.qmatmul(w, x, qh.FLAG_FORCE_MATVEC)
    # rows apart, so that one wrong tile cannot hide in the rest
    err = (got - want).double().norm(dim=1) / want.double().norm(dim=1)
    assert err.max().item() <= 4 * (k // block) * 2.0 ** -24 + 2e-7, err.max().item()
