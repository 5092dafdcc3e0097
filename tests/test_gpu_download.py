"""GGML blocks back on the host: sizes on both sides of the line where the download goes piece by piece, whole pieces and ragged last ones, into
pinned memory, and from several threads at once."""
import ctypes as C
import threading

import numpy as np
import pytest
import torch

from oracle import cpu_oracle as orc
from tests.test_gpu_fused_neighbours import qh  # noqa: F401

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def weight(qh, dt, nblocks, seed):  # noqa: F811
    blocks = np.random.default_rng(seed).integers(0, 256, nblocks * orc.TYPE_SIZE[dt], dtype=np.uint8)
    return qh.QWeight.from_ggml_flat(dt, blocks, 0), blocks


@pytest.mark.parametrize("dt,nblocks", [(orc.Q8_0, 1), (orc.Q8_0, 5 * MIB // 34), (orc.Q8_0, 5 * MIB // 34 + 1), (orc.Q4K, 8 * MIB // 144 + 1),
                                        (orc.Q6K, 10 * MIB // 210 + 1), (orc.Q4_0, 33 * MIB // 18), (orc.Q5K, 9 * MIB // 11), (orc.Q5K, MIB * 16 // 176 * 11)])
def test_same_bytes(qh, dt, nblocks):  # noqa: F811
    w, blocks = weight(qh, dt, nblocks, nblocks)
    assert np.array_equal(w.to_ggml(), blocks)
    pinned = torch.empty(blocks.size, dtype=torch.uint8, pin_memory=True)
    qh.check(qh.load().cq_weight_to_ggml(w.handle, C.c_void_p(pinned.data_ptr()), blocks.size))
    assert np.array_equal(pinned.numpy(), blocks)
    guarded = np.full(blocks.size + 16, 7, dtype=np.uint8)   # an odd address, nothing written past the end
    qh.check(qh.load().cq_weight_to_ggml(w.handle, C.c_void_p(guarded.ctypes.data + 1), blocks.size))
    assert np.array_equal(guarded[1:blocks.size + 1], blocks) and guarded[0] == 7 and (guarded[blocks.size + 1:] == 7).all()


@pytest.mark.parametrize("dt", [orc.Q4_1, orc.Q5_0, orc.Q5_1, orc.Q2K, orc.Q3K, orc.Q8_0, orc.Q6K])
@pytest.mark.parametrize("nblocks", [1, 7, 300])
def test_zeros_and_quantized_into_them(qh, dt, nblocks):  # noqa: F811
    bs = orc.BLOCK_SIZE[dt]
    w = qh.QWeight.zeros_flat(dt, nblocks * bs)
    assert not w.to_ggml().any() and not w.dequantize().cpu().numpy().any()
    x = np.random.default_rng(nblocks).standard_normal(nblocks * bs).astype(np.float32)
    side = torch.cuda.Stream()
    xd = torch.from_numpy(x).cuda()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        w.quantize_(xd)
    assert np.array_equal(w.to_ggml(), orc.quantize(dt, x.reshape(1, -1)))


def test_threads(qh):  # noqa: F811
    made = [weight(qh, orc.Q8_0, (6 + i) * MIB // 34, i) for i in range(3)]
    same = [0] * 3

    def run(i):
        for _ in range(4):
            same[i] += int(np.array_equal(made[i][0].to_ggml(), made[i][1]))

    threads = [threading.Thread(target=run, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert same == [4, 4, 4]
