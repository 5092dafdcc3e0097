"""Two to four rows of small K-quant weights by the split-K kernel that quantizes the rows itself: around the sizes where it takes them
(blocks of a row no multiple of four, 2048 elements, 4096 weight rows, two rows), and the rows that it leaves in the workspace."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle as orc  # noqa: E402
from test_gpu_fused_neighbours import qh  # noqa: E402,F401
from test_gpu_parity import check_f32, dev, make_inputs  # noqa: E402


@pytest.mark.parametrize("dt", [orc.Q4K, orc.Q5K, orc.Q6K, orc.Q3K])
@pytest.mark.parametrize("m,k,n", [(2, 256, 16), (2, 768, 4096), (2, 1280, 77), (3, 1792, 4096), (3, 1792, 4097), (3, 2304, 40), (3, 768, 17), (4, 768, 300)])
def test_small_weights(qh, dt, m, k, n):  # noqa: F811
    w, x = make_inputs(dt + m + k + n, m, k, n)
    blocks = orc.quantize(dt, w)
    qw = qh.QWeight.from_ggml(dt, blocks, n, k)
    check_f32(qh.qmatmul(qw, dev(x)).cpu().numpy(), orc.matmul(dt, x, blocks, n))
    for y in qh.qmatmul_multi([qw, qw], dev(x)):
        check_f32(y.cpu().numpy(), orc.matmul(dt, x, blocks, n))


@pytest.mark.parametrize("m", [2, 3])
def test_the_rows_are_left_in_the_workspace(qh, m):  # noqa: F811
    k, n = 768, 64
    w, x = make_inputs(m, m, k, n)
    qw = qh.QWeight.from_ggml(orc.Q4K, orc.quantize(orc.Q4K, w), n, k)
    L, xd = qh.load(), dev(x)
    ws = torch.zeros(L.cq_workspace_bytes(qw.handle, m, 0), dtype=torch.uint8, device="cuda")
    ys = [torch.empty((m, n), dtype=torch.float32, device="cuda") for _ in range(2)]
    for y, flags in zip(ys, (0, qh.FLAG_REUSE_ACT)):
        assert L.cq_qmatmul(qw.handle, C.c_void_p(xd.data_ptr()), m, C.c_void_p(y.data_ptr()), flags, C.c_void_p(ws.data_ptr()), ws.numel(), None) == 0
    torch.cuda.synchronize()
    err = (ys[0] - ys[1]).norm() / ys[0].norm()
    assert err.item() <= 4 * 3 * 2.0 ** -24   # the same products, three blocks a row in any order
