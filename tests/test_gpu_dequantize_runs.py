"""Dequantized results leave a wave as one run of the output: block counts around the ends of waves (2048 elements, 1024 of the types held
as Q8_0) and workgroups, nothing written past the end, the bits of the oracle."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import cpu_oracle as orc
from tests.test_gpu_fused_neighbours import qh  # noqa: F401

pytestmark = pytest.mark.gpu

TYPES = [orc.Q4_0, orc.Q4_1, orc.Q5_0, orc.Q5_1, orc.Q8_0, orc.Q2K, orc.Q3K, orc.Q4K, orc.Q5K, orc.Q6K]


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("elements", [256, 768, 1024, 1280, 2048, 2304, 4096, 8192 - 256, 8192, 8192 + 256, 32768 + 1792])
def test_runs_and_their_ends(qh, dt, elements):  # noqa: F811
    counts = [elements] if orc.BLOCK_SIZE[dt] == 256 else [elements, elements + 32, elements + 32 * 7, elements - 32]
    for n in counts:
        x = np.random.default_rng(n).standard_normal(n).astype(np.float32)
        blocks = orc.quantize(dt, x.reshape(1, -1))
        w = qh.QWeight.from_ggml_flat(dt, blocks, 0)
        want = orc.dequantize(dt, blocks).ravel()
        for dtype, call, wanted in ((torch.float32, "cq_weight_dequantize", want), (torch.float16, "cq_weight_dequantize_f16", want.astype(np.float16))):
            out = torch.full((n + 64,), 7.0, dtype=dtype, device="cuda")
            qh.check(getattr(qh.load(), call)(w.handle, C.c_void_p(out.data_ptr()), None))
            torch.cuda.synchronize()
            got = out.cpu().numpy()
            assert np.array_equal(got[:n].view(np.uint8), wanted.view(np.uint8)), (n, call)
            assert (got[n:] == 7.0).all(), (n, call)


@pytest.mark.parametrize("dt,half", [(orc.Q4_0, True), (orc.Q8_0, True), (orc.Q4_1, False), (orc.Q4K, True), (orc.Q5K, False), (orc.Q6K, False), (orc.Q2K, True)])
def test_results_around_the_size_of_streamed_ones(qh, dt, half):  # noqa: F811
    """240 MB of results and more are stored non-temporal: the bits of the same blocks dequantized in smaller parts, on both sides of the line."""
    k = 4096
    line = 240_000_000 // (k * (2 if half else 4))
    for n in (line, line + 1):
        g = torch.Generator(device="cuda").manual_seed(n)
        w = qh.QWeight.zeros(dt, n, k).quantize_(torch.randn(n, k, generator=g, device="cuda"))
        got = w.dequantize_f16() if half else w.dequantize()
        blocks = w.to_ggml().reshape(n, -1)
        for lo in range(0, n, 8192):
            part = blocks[lo:lo + 8192]
            v = qh.QWeight.from_ggml(dt, part.ravel(), len(part), k)
            assert torch.equal(got[lo:lo + 8192], v.dequantize_f16() if half else v.dequantize()), lo
        del w, got
