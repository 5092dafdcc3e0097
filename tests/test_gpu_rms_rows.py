"""rms_norm in front of two to four rows in the one-launch decode kernel: a row's bits are those of its own one-row call (the same
sums in the same order), for one weight and for several, at one to four passes of a wave over the row, full and partly filled."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle as orc  # noqa: E402
from test_gpu_parity import check_f32, dev, make_inputs  # noqa: E402


@pytest.fixture(scope="module")
def qh():
    from candle_amd import qhip
    qhip.load()
    assert qhip.load().cq_device_count() >= 1, "no HIP device visible"
    return qhip


@pytest.mark.parametrize("dt,m,k", [
    (orc.Q4K, 2, 256), (orc.Q4K, 3, 3840), (orc.Q4K, 4, 4096), (orc.Q4K, 2, 4352), (orc.Q4K, 3, 8192), (orc.Q4K, 2, 16384),
    (orc.Q5K, 4, 4096), (orc.Q5K, 2, 12032), (orc.Q6K, 2, 512), (orc.Q6K, 4, 3072), (orc.Q6K, 4, 4096), (orc.Q6K, 3, 5888),
    (orc.Q6K, 3, 8192), (orc.Q3K, 2, 1024), (orc.Q3K, 4, 4096)])
@pytest.mark.parametrize("ns", [(8,), (77,), (9, 40, 131), (300, 16)])
def test_rows_equal_their_one_row_calls(qh, dt, m, k, ns):
    rng = np.random.default_rng(k + m + len(ns))
    x = rng.standard_normal((m, k)).astype(np.float32) * np.float32([[1e-3], [7.0], [1.0], [300.0]])[:m]
    alpha = rng.standard_normal(k).astype(np.float32)
    blocks = [orc.quantize(dt, make_inputs(k + i, 1, k, n)[0]) for i, n in enumerate(ns)]
    ws = [qh.QWeight.from_ggml(dt, b, n, k) for b, n in zip(blocks, ns)]
    xd, ad = dev(x), dev(alpha)
    kw = dict(pre=qh.PRE_RMS_NORM, aux=ad, eps=1e-5)
    outs = qh.qmatmul_multi(ws, xd, **kw) if len(ws) > 1 else [qh.qmatmul(ws[0], xd, **kw)]
    for w, b, y in zip(ws, blocks, outs):
        for r in range(m):
            assert torch.equal(y[r:r + 1], qh.qmatmul(w, xd[r:r + 1].contiguous(), **kw))
        check_f32(y.cpu().numpy(), orc.matmul(dt, orc.rms_norm(x, alpha, 1e-5), b, w.shape[0]))


def test_a_reused_workspace_follows_more_than_three_weights(qh):
    """Four weights: no launch over all of them, so the first call leaves its rows in the workspace for the others."""
    k, m = 1024, 2
    rng = np.random.default_rng(3)
    x, alpha = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal(k).astype(np.float32)
    blocks = [orc.quantize(orc.Q4K, make_inputs(i, 1, k, 48)[0]) for i in range(4)]
    ws = [qh.QWeight.from_ggml(orc.Q4K, b, 48, k) for b in blocks]
    for b, y in zip(blocks, qh.qmatmul_multi(ws, dev(x), pre=qh.PRE_RMS_NORM, aux=dev(alpha), eps=1e-5)):
        check_f32(y.cpu().numpy(), orc.matmul(orc.Q4K, orc.rms_norm(x, alpha, 1e-5), b, 48))


def test_weights_that_decide_apart(qh):
    """One weight of many rows and two of few: two launches together, the one launch for the small ones alone.  The outputs agree to the order of
    the sums."""
    k, m, ns = 512, 2, (8192, 1024, 1024)
    rng = np.random.default_rng(5)
    x, alpha = dev(rng.standard_normal((m, k)).astype(np.float32)), dev(rng.standard_normal(k).astype(np.float32))
    ws = [qh.QWeight.from_ggml(orc.Q4K, orc.quantize(orc.Q4K, make_inputs(i, 1, k, n)[0]), n, k) for i, n in enumerate(ns)]
    f = qh.load()._Z34cq_matvec_fused_rms_rows_supportedPKPK9cq_weightil
    f.restype, f.argtypes = C.c_bool, [C.c_void_p, C.c_int, C.c_int64]
    assert not f((C.c_void_p * 3)(*(w.handle.value for w in ws)), 3, m) and f((C.c_void_p * 1)(ws[1].handle.value), 1, m)
    kw = dict(pre=qh.PRE_RMS_NORM, aux=alpha, eps=1e-5)
    for w, y in zip(ws, qh.qmatmul_multi(ws, x, **kw)):
        own = qh.qmatmul(w, x, **kw)
        # (the one launch scales the results, the quantizer its input: a quant beside the middle of two may go the other way)
        assert ((y - own).norm() / own.norm()).item() <= 2e-3


@pytest.mark.parametrize("dt,m,k,ns", [(orc.Q4K, 2, 768, (40,)), (orc.Q4K, 3, 4096, (64, 16)), (orc.Q4K, 4, 4096, (64,)), (orc.Q5K, 3, 2048, (33, 20)),
                                       (orc.Q6K, 4, 3072, (48, 16, 8)), (orc.Q6K, 3, 5888, (40,))])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), 1e30, 0.0])
def test_a_bad_row_stays_alone(qh, dt, m, k, ns, bad):
    """A row with a NaN, an infinity, squares beyond f32, or of zeros only, first, in the middle and last: its own one-row call's bits, and the
    finite rows beside it theirs."""
    rng = np.random.default_rng(k + m)
    alpha = dev(rng.standard_normal(k).astype(np.float32))
    ws = [qh.QWeight.from_ggml(dt, orc.quantize(dt, make_inputs(k + i, 1, k, n)[0]), n, k) for i, n in enumerate(ns)]
    kw = dict(pre=qh.PRE_RMS_NORM, aux=alpha, eps=1e-5)
    for at in range(m):
        x = rng.standard_normal((m, k)).astype(np.float32)
        if bad == 0.0:
            x[at] = 0.0
        else:
            x[at, k // 2 + 3] = bad
        xd = dev(x)
        outs = qh.qmatmul_multi(ws, xd, **kw) if len(ws) > 1 else [qh.qmatmul(ws[0], xd, **kw)]
        for w, y in zip(ws, outs):
            for r in range(m):
                one = qh.qmatmul(w, xd[r:r + 1].contiguous(), **kw)
                assert torch.equal(y[r:r + 1].view(torch.int32), one.view(torch.int32)), (at, r)
                assert r == at or (bool(torch.isfinite(one).all()) and bool((one != 0).any()))


@pytest.mark.parametrize("m", [2, 3, 4])
def test_the_workspace_is_asked_for(qh, m):
    """Several weights behind rms_norm in one launch: a missing or short workspace is refused, as where the rows go through it."""
    k = 1024
    w = qh.QWeight.from_ggml(orc.Q4K, orc.quantize(orc.Q4K, make_inputs(m, 1, k, 48)[0]), 48, k)
    L, x, alpha = qh.load(), dev(np.ones((m, k), np.float32)), dev(np.ones(k, np.float32))
    ys = [torch.full((m, 48), 7.0, device="cuda") for _ in range(2)]
    need = L.cq_workspace_bytes(w.handle, m, 0)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    handles, outs = (C.c_void_p * 2)(w.handle.value, w.handle.value), (C.c_void_p * 2)(*(y.data_ptr() for y in ys))
    for room, size in ((None, need), (ws.data_ptr(), need - 1)):
        assert L.cq_qmatmul_multi(handles, 2, qh.PRE_RMS_NORM, C.c_void_p(x.data_ptr()), C.c_void_p(alpha.data_ptr()), 1e-5, m, outs, 0, room, size, None) == -4
    torch.cuda.synchronize()
    assert all(bool((y == 7.0).all()) for y in ys)
