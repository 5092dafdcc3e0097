"""Two and three rows of small K-quant weights, also with rows of no multiple of four blocks: the one launch of dot products, alone and over several
weights, so that every row has the bits of its own one-row call and every output of cq_qmatmul_multi those of its weight's own call."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle as orc  # noqa: E402
from test_gpu_fused_neighbours import qh  # noqa: E402,F401
from test_gpu_parity import check_f32, dev, make_inputs  # noqa: E402


@pytest.mark.parametrize("dt", [orc.Q4K, orc.Q5K, orc.Q6K, orc.Q3K])
@pytest.mark.parametrize("m,k,ns", [(2, 256, (16, 40)), (2, 768, (4096, 64)), (2, 1280, (77, 300)), (3, 768, (64, 17, 40)), (3, 1024, (300, 64)),
                                    (3, 1792, (2048, 33)), (3, 2304, (40, 48)), (4, 1024, (64, 300))])
def test_rows_and_outputs_are_those_of_their_own_calls(qh, dt, m, k, ns):  # noqa: F811
    x = make_inputs(dt + m + k, m, k, 1)[1]
    blocks = [orc.quantize(dt, make_inputs(k + i, 1, k, n)[0]) for i, n in enumerate(ns)]
    ws = [qh.QWeight.from_ggml(dt, b, n, k) for b, n in zip(blocks, ns)]
    xd = dev(x)
    for w, b, n, y in zip(ws, blocks, ns, qh.qmatmul_multi(ws, xd)):
        assert torch.equal(y, qh.qmatmul(w, xd))
        for r in range(m):
            assert torch.equal(y[r:r + 1], qh.qmatmul(w, xd[r:r + 1].contiguous()))
        check_f32(y.cpu().numpy(), orc.matmul(dt, x, b, n))
