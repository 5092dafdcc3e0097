"""The matrix-core kernels on weights that are no whole number of tiles: row counts around 16 and 32, rows of an even number
of 32-element blocks that is no multiple of eight, every row-group count of the split-K kernel, launches that split K."""
import numpy as np
import pytest

from oracle import cpu_oracle as orc

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def check(got, want):
    got = got.cpu().numpy().astype(np.float64)
    for r in range(want.shape[0]):
        ref = np.linalg.norm(want[r].astype(np.float64))
        assert np.linalg.norm(got[r] - want[r]) <= 1e-5 * ref, (r, np.linalg.norm(got[r] - want[r]) / ref)


def inputs(seed, m, k, n):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((n, k)) * 0.02).astype(np.float32), rng.standard_normal((m, k)).astype(np.float32)


@pytest.mark.parametrize("dt", [orc.Q4K, orc.Q5K, orc.Q6K])
@pytest.mark.parametrize("m,k,n", [(2, 256, 17), (8, 4096, 31), (16, 2304, 47), (24, 768, 33), (31, 1024, 127), (40, 512, 129), (5, 3072, 4113),
                                   (70, 1280, 255), (33, 4096, 300), (130, 2048, 1027), (200, 6144, 131), (9, 4096, 4099), (129, 768, 2305)])
def test_kquants(dt, m, k, n):
    from candle_amd import qhip
    w, x = inputs(m + k + n, m, k, n)
    blocks = orc.quantize(dt, w)
    y = qhip.qmatmul(qhip.QWeight.from_ggml(dt, blocks, n, k), torch.from_numpy(x).cuda())
    check(y, orc.matmul(dt, x, blocks, n))


@pytest.mark.parametrize("dt", [orc.Q4_0, orc.Q8_0, orc.Q5_0, orc.Q5_1])
@pytest.mark.parametrize("m,k,n", [(5, 320, 16), (8, 576, 17), (16, 3264, 47), (12, 4032, 4113), (24, 832, 31), (17, 256, 131), (33, 448, 129), (40, 64, 40),
                                   (70, 3200, 255), (130, 960, 1027), (200, 4160, 131), (15, 4160, 100), (129, 704, 2305), (31, 576, 96)])
def test_blocks_of_32(dt, m, k, n):
    from candle_amd import qhip
    w, x = inputs(m + k + n, m, k, n)
    blocks = orc.quantize(dt, w)
    y = qhip.qmatmul(qhip.QWeight.from_ggml(dt, blocks, n, k), torch.from_numpy(x).cuda())
    check(y, orc.matmul(dt, x, blocks, n))


@pytest.mark.parametrize("m", [6, 40])
def test_short_last_step_keeps_rows_apart(m):
    """What follows a row in memory is copied with its last, shorter K step: an infinity there must not reach the row."""
    from candle_amd import qhip
    k, n = 320, 160
    w, x = inputs(m, m, k, n)
    blocks = orc.quantize(orc.Q8_0, w)
    qw = qhip.QWeight.from_ggml(orc.Q8_0, blocks, n, k)
    bad = x.copy()
    bad[3, 5] = np.inf
    y, yb = qhip.qmatmul(qw, torch.from_numpy(x).cuda()), qhip.qmatmul(qw, torch.from_numpy(bad).cuda())
    keep = [r for r in range(m) if r != 3]
    assert torch.allclose(y[keep], yb[keep], rtol=1e-5, atol=1e-5)
