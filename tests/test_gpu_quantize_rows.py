"""Q8K quantizer of many rows (a block per sixteen lanes) against the kernel of few rows (a block per wave), which the oracle
tests pin: the same bytes, also where both signs reach the largest |x|, and for zeros, NaN, infinities and tiny blocks."""
import numpy as np
import pytest
import torch

from oracle import cpu_oracle as orc
from tests.test_gpu_fused_neighbours import dev, qh  # noqa: F401

pytestmark = pytest.mark.gpu


def rows(m, k):
    rng = np.random.default_rng(m + k)
    x = rng.standard_normal((m, k)).astype(np.float32) * np.exp(rng.uniform(-60, 60, (m, 1))).astype(np.float32)
    blocks = x.reshape(-1, 256)
    for i, b in enumerate(blocks):
        top = np.float32(1.5) * np.abs(b).max()
        at = rng.choice(256, 2, replace=False)
        kind = i % 9
        if kind == 0:
            b[at] = top, -top           # a tie of both signs, in either order
        elif kind == 1:
            b[at] = top                 # of one sign
        elif kind == 2:
            b[at[0] // 4 * 4:at[0] // 4 * 4 + 4] = -top, top, top, -top   # inside one lane
        elif kind == 3:
            b[:] = 0.0 if i % 2 else -0.0
        elif kind == 4:
            b[at[0]] = np.nan
        elif kind == 5:
            b[at] = np.inf, -np.inf
        elif kind == 6:
            b[:] *= np.float32(1e-38) / top   # 128 / max overflows
    return x


@pytest.mark.parametrize("m,k", [(1024, 256), (205, 1280), (33, 8192), (90, 3072)])
@pytest.mark.parametrize("silu", [False, True])
def test_many_rows_give_the_bytes_of_few(qh, m, k, silu):  # noqa: F811
    x = rows(m, k)
    args = (qh.PRE_SILU_MUL, dev(rows(m, k)[::-1].copy())) if silu else ()
    xd = dev(x)
    got = qh.quantize_act(orc.Q8K, xd, *args)
    step = 7   # far fewer blocks than the other kernel begins at
    few = [qh.quantize_act(orc.Q8K, xd[i:i + step].contiguous(), *((args[0], args[1][i:i + step].contiguous()) if silu else ()))
           for i in range(0, m, step)]
    assert torch.equal(got.reshape(-1), torch.cat([f.reshape(-1) for f in few]))
    if not silu:
        blocks = x.reshape(-1, 256)   # (a row's blocks are independent)
        ok = np.isfinite(blocks).all(1)
        want = np.stack([orc.quantize(orc.Q8K, b) for b in blocks[ok]])
        assert np.array_equal(got.cpu().numpy().reshape(len(blocks), -1)[ok], want)


@pytest.mark.parametrize("dt", [orc.Q4K, orc.Q5K, orc.Q6K])
@pytest.mark.parametrize("k", [256, 2304, 4096, 16384])
def test_one_row_gives_the_bits_of_its_quantized_row(qh, dt, k):  # noqa: F811
    """The one-launch kernels quantize their row in code of their own: on such blocks too the bits of the call that goes through the quantizer."""
    blocks = orc.quantize(dt, np.random.default_rng(k).standard_normal((24, k)).astype(np.float32) * np.float32(0.02))
    w = qh.QWeight.from_ggml(dt, blocks, 24, k)
    for row in rows(11, k):
        x = dev(row[None])
        one, staged = qh.qmatmul(w, x), qh.qmatmul(w, x, qh.FLAG_STAGED_ACT)
        assert torch.equal(one.view(torch.int32), staged.view(torch.int32))
