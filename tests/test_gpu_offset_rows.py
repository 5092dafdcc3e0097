"""Q4_1 / Q5_1 / Q2K with two to four rows on either side of the line between the one-launch kernel and the split-K kernel, by the row
count, the weight rows and the row length: both sides against the oracle, and the one launch by its bits, those of one-row calls."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle as orc  # noqa: E402
from test_gpu_fused_neighbours import qh  # noqa: E402,F401
from test_gpu_parity import check_f32, dev, make_inputs  # noqa: E402


@pytest.mark.parametrize("dt,m,k,n", [
    (orc.Q2K, 2, 512, 8000), (orc.Q2K, 3, 512, 4100), (orc.Q2K, 3, 512, 8000), (orc.Q2K, 4, 256, 40), (orc.Q2K, 4, 2048, 264),
    (orc.Q2K, 2, 8192, 33), (orc.Q2K, 2, 8448, 1024), (orc.Q2K, 2, 8448, 1025), (orc.Q4_1, 4, 512, 4100), (orc.Q4_1, 4, 512, 9000),
    (orc.Q5_1, 3, 768, 9000), (orc.Q4_1, 2, 512, 16400)])
def test_either_side_of_the_line(qh, dt, m, k, n):  # noqa: F811
    w, x = make_inputs(dt + m + k + n, m, k, n)
    blocks = orc.quantize(dt, w + 0.5 * abs(w).mean())   # offsets that matter
    qw = qh.QWeight.from_ggml(dt, blocks, n, k)
    got = qh.qmatmul(qw, dev(x))
    check_f32(got.cpu().numpy(), orc.matmul(dt, x, blocks, n))
    one_launch = qh.load()._Z30cq_matvec_fused_rows_supportedPK9cq_weightl
    one_launch.restype, one_launch.argtypes = C.c_bool, [C.c_void_p, C.c_int64]
    rows = torch.cat([qh.qmatmul(qw, dev(x[r:r + 1])) for r in range(m)])
    assert torch.equal(got, rows) == one_launch(qw.handle, m)   # (a row of split K differs somewhere among its columns)
    outs = qh.qmatmul_multi([qw, qw], dev(x))   # (shares the quantized rows where a single call does not take them in one launch)
    for y in outs:
        check_f32(y.cpu().numpy(), orc.matmul(dt, x, blocks, n))
