"""Rows of a small weight: the launch whose waves quantize the rows they contract.  The same bits as the quantizer launch and the split-K
launch after it (CQ_FLAG_STAGED_ACT asks for the two), in y and in the workspace, also for rows of zeros, infinities and NaN and for a block
whose largest magnitude comes with both signs.  The workspace is read back through calls that reuse it: the split-K kernel and the dot-product
kernel, which between them read every plane the quantizer writes."""
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_fused_neighbours import qh  # noqa: F401

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    return torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("dt,n,k,m", [("Q4K", 16, 256, 5), ("Q4K", 4096, 1024, 8), ("Q4K", 1000, 768, 4), ("Q5K", 1031, 768, 7), ("Q6K", 33, 512, 5),
                                      ("Q6K", 4090, 256, 4), ("Q3K", 512, 1024, 6), ("Q2K", 300, 512, 5), ("Q4K", 2048, 2048, 16), ("Q5K", 300, 1792, 37), ("Q6K", 16, 1024, 255), ("Q3K", 65, 256, 9),
                                      ("Q8_0", 16, 256, 5), ("Q8_0", 4096, 1024, 8),
                                      ("Q4_0", 1000, 320, 7), ("Q4_0", 4095, 960, 6), ("Q4_1", 500, 704, 5), ("Q5_1", 129, 1024, 7)])
def test_same_bits_as_two_launches(qh, dt, n, k, m):  # noqa: F811
    g = torch.Generator(device="cuda").manual_seed(n + k + m)
    w = QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.05, GgmlDType[dt]).weight
    x = torch.randn(m, k, generator=g, device="cuda")
    x[0, :256] = 0.0
    x[1, 40], x[1, 200] = -9.0, 9.0
    x[2, 17], x[2, 70] = 9.0, -9.0
    bad = x.clone()
    bad[1, 3], bad[m - 1, k - 1] = float("nan"), float("inf")
    for rows in (x, bad):
        ws, ws2 = qh.Workspace(), qh.Workspace()
        y = torch.full((m + 1, n), 7.0, device="cuda")
        qh.qmatmul(w, rows, out=y[:m], workspace=ws)
        two = qh.qmatmul(w, rows, flags=qh.FLAG_STAGED_ACT, workspace=ws2)
        assert same_bits(y[:m], two) and bool((y[m] == 7.0).all())
        if m > 4:   # (up to four rows may be one launch that leaves the workspace alone)
            for flags in (qh.FLAG_REUSE_ACT, qh.FLAG_REUSE_ACT | qh.FLAG_FORCE_MATVEC):
                reused = [qh.qmatmul(w, torch.zeros_like(x), flags=flags, workspace=v) for v in (ws, ws2)]
                assert same_bits(reused[0], reused[1])
                if not flags & qh.FLAG_FORCE_MATVEC:
                    assert same_bits(reused[0], two)
