"""Weights without rows among those of cq_qmatmul_multi: the first weight that has rows quantizes the shared activations, wherever it stands."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle as orc  # noqa: E402
from test_gpu_fused_neighbours import qh  # noqa: E402,F401
from test_gpu_parity import check_f32, dev, make_inputs  # noqa: E402


@pytest.mark.parametrize("dt", [orc.Q4K, orc.Q8_0, orc.Q4_1, orc.Q2K])
@pytest.mark.parametrize("m", [1, 2, 7, 40, 130])
@pytest.mark.parametrize("ns", [(0, 64, 40), (64, 0, 40), (0, 0, 33), (0, 0)])
def test_outputs_beside_empty_weights(qh, dt, m, ns):  # noqa: F811
    k = 1024
    x, aux = make_inputs(m + dt, m, k, 1)[1], dev(make_inputs(m, 1, k, 1)[1][0])
    blocks = [orc.quantize(dt, make_inputs(k + i, 1, k, n)[0]) if n else None for i, n in enumerate(ns)]
    ws = [qh.QWeight.from_ggml(dt, b, n, k) if n else qh.QWeight.zeros(dt, 0, k) for b, n in zip(blocks, ns)]
    for pre in (qh.PRE_NONE, qh.PRE_RMS_NORM):
        kw = dict(pre=pre, aux=aux if pre else None, eps=1e-5)
        stale = qh.Workspace()
        stale.get(1 << 20, torch.device("cuda", 0)).zero_()   # a call that trusts it gives zeros
        for w, b, n, y in zip(ws, blocks, ns, qh.qmatmul_multi(ws, dev(x), workspace=stale, **kw)):
            assert y.shape == (m, n)
            if n:
                own = qh.qmatmul(w, dev(x), **kw)
                assert (y - own).norm().item() <= 4 * (k // 32) * 2.0 ** -24 * own.norm().item()   # the row's blocks in another order
                if pre == qh.PRE_NONE:
                    check_f32(y.cpu().numpy(), orc.matmul(dt, x, b, n))
