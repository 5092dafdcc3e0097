"""The device weight quantizers where their work split can go wrong: block counts around a workgroup's, rows that start
off a 16-byte boundary, and values their rounding has to clamp (infinities, NaN, magnitudes far beyond a quant)."""
import numpy as np
import pytest

from oracle import cpu_oracle as orc

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TYPES = [orc.Q4_0, orc.Q4_1, orc.Q5_0, orc.Q5_1, orc.Q8_0, orc.Q2K, orc.Q3K, orc.Q4K, orc.Q5K, orc.Q6K]


def _values(rng, count):
    x = (rng.standard_normal(count) * 0.02).astype(np.float32)
    x *= np.repeat(10.0 ** rng.uniform(-6, 3, -(-count // 64)), 64)[:count].astype(np.float32)
    x[rng.random(count) < 0.01] = 0.0
    x[rng.random(count) < 0.01] = -0.0
    return x


# a workgroup takes 256 groups: 256 blocks of 32 elements, 32 or 16 blocks of 256
@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("blocks", [1, 15, 16, 17, 32, 33, 255, 257])
def test_block_counts(dt, blocks):
    from candle_amd import qhip
    k = orc.BLOCK_SIZE[dt]
    w = _values(np.random.default_rng(1000 * dt + blocks), blocks * k).reshape(blocks, k)
    src = torch.empty(w.size + 1, device="cuda")[1:]   # not 16-byte aligned
    src.copy_(torch.from_numpy(w.reshape(-1)))
    qw = qhip.QWeight.zeros(dt, blocks, k)
    qw.quantize_(src)
    assert np.array_equal(qw.to_ggml(), orc.quantize(dt, w))


@pytest.mark.parametrize("dt", TYPES)
def test_extreme_values(dt):
    from candle_amd import qhip
    n, k = 40, 512
    rng = np.random.default_rng(dt)
    w = _values(rng, n * k).reshape(n, k)
    w[0, ::5] = 3e38
    w[1, ::7] = -3e38
    w[2] = 1e-42 * rng.integers(-9, 10, k)
    w[3, 3::16] = np.inf
    w[4, 5::32] = -np.inf
    w[5, 9::16] = np.nan
    w[6, ::16] = np.nan
    w[7] = np.nan
    w[8] = rng.integers(-3, 4, k) * 0.5
    qw = qhip.QWeight.zeros(dt, n, k)
    qw.quantize_(torch.from_numpy(w).cuda())
    assert np.array_equal(qw.to_ggml(), orc.quantize(dt, w))
