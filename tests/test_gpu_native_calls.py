"""The native side of qhip's calls (csrc/calls.cpp) on the device: what it takes and what it refuses."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle as orc  # noqa: E402  (checker only)
from test_gpu_parity import check_f32, dev, make_inputs  # noqa: E402


@pytest.fixture(scope="module")
def qh():
    from candle_amd import qhip
    qhip.load()
    assert qhip.load().cq_device_count() >= 1, "no HIP device visible"
    return qhip


@pytest.mark.parametrize("dt", [orc.Q4K, orc.Q8_0])
def test_three_hundred_experts(qh, dt):
    """More experts than any launch's table holds: a launch per expert, as the C ABI has it."""
    n, k, experts = 32, 256, 300
    blocks = [orc.quantize(dt, make_inputs(e, 1, k, n)[0]) for e in range(8)]
    ws = [qh.QWeight.from_ggml(dt, b, n, k) for b in blocks]
    x = np.random.default_rng(1).standard_normal((16, k)).astype(np.float32)
    counts = np.zeros(experts, np.int64)
    counts[[0, 5, 255, 256, 257, 299]] = [2, 3, 1, 4, 1, 5]
    offsets = np.concatenate([[0], counts.cumsum()]).astype(np.int32)
    y = qh.qmatmul_grouped([ws[e % 8] for e in range(experts)], dev(x), None, offsets).cpu().numpy()
    for e in np.flatnonzero(counts):
        lo, hi = offsets[e], offsets[e + 1]
        check_f32(y[lo:hi], orc.matmul(dt, x[lo:hi], blocks[e % 8], n))


def test_many_weights_on_the_same_rows(qh):
    n, k = 32, 256
    ws = [qh.QWeight.from_ggml(orc.Q4K, orc.quantize(orc.Q4K, make_inputs(e, 1, k, n)[0]), n, k) for e in range(3)]
    x = dev(np.random.default_rng(2).standard_normal((2, k)).astype(np.float32))
    want = [qh.qmatmul(w, x) for w in ws]
    for i, y in enumerate(qh.qmatmul_multi([ws[i % 3] for i in range(260)], x)):
        assert torch.equal(y, want[i % 3])


def weight(qh, n=64, k=512):
    return qh.QWeight.from_ggml(orc.Q4K, orc.quantize(orc.Q4K, make_inputs(7, 1, k, n)[0]), n, k)


def test_refused_arguments(qh):
    """What the calls refuse, each in its own words; the call after it runs."""
    w, k = weight(qh), 512
    x = torch.ones(4, k, device="cuda")
    alpha = torch.ones(k, device="cuda")
    want = qh.qmatmul(w, x)
    offsets = np.array([0, 4], np.int32)
    for bad, words in ((x.cpu(), "device tensor"), (x.half(), "f32"), (torch.ones(k, 4, device="cuda").t(), "not contiguous"),
                       (x[:, :256].contiguous(), "incompatible"), (x[0], "only one dimension")):
        with pytest.raises(qh.QHipError, match=words):
            qh.qmatmul(w, bad)
        with pytest.raises(qh.QHipError, match=words):
            qh.qmatmul_multi([w, w], bad)
        if words in ("device tensor", "f32", "not contiguous"):
            with pytest.raises(qh.QHipError, match=words):
                qh.qmatmul_grouped([w], bad, None, offsets)
    for pre, aux, words in ((qh.PRE_RMS_NORM, alpha[:256].contiguous(), "rms-norm"), (qh.PRE_RMS_NORM, x, "rms-norm"),
                            (qh.PRE_SILU_MUL, alpha, "silu-mul"), (qh.PRE_SILU_MUL, x.double(), "f32"), (9, alpha, "unknown fused step")):
        for call in (lambda: qh.qmatmul(w, x, pre=pre, aux=aux), lambda: qh.qmatmul_multi([w, w], x, pre=pre, aux=aux),
                     lambda: qh.qmatmul_grouped([w], x, None, offsets, pre=pre, aux=aux)):
            with pytest.raises(qh.QHipError, match=words):
                call()
    for bad_offsets in (offsets[:1], np.array([0, -1], np.int32), np.array([1, 4], np.int32), np.array([0, 5, 4], np.int32)):
        with pytest.raises((qh.QHipError, RuntimeError)):
            qh.qmatmul_grouped([w, w][: max(1, len(bad_offsets) - 1)], x, None, bad_offsets)
    with pytest.raises(qh.QHipError):
        qh.qmatmul_grouped([], x, None, offsets)
    assert torch.equal(qh.qmatmul(w, x), want)


def test_function_transforms_are_refused(qh):
    """vmap and grad hand over tensors without memory: an error, and the process goes on."""
    from candle_amd.quantized import QMatMul, QTensor
    w = weight(qh)
    mat = QMatMul(QTensor(w, w.shape))
    x = torch.ones(3, 2, 512, device="cuda")
    want = mat.forward(x)
    for call in (mat.forward, lambda v: qh.qmatmul_multi([w, w], v)[0], lambda v: qh.qmatmul_grouped([w], v, None, np.array([0, 2], np.int32))):
        with pytest.raises(RuntimeError):
            torch.func.vmap(call)(x)
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda v: call(v).sum())(x[0])
    assert torch.equal(mat.forward(x), want)


def test_calls_run_on_the_current_stream(qh):
    """Inputs still being written on another stream, the calls behind them on that stream, nothing waited for in between."""
    w, k = weight(qh), 512
    src = torch.randn(8, k, device="cuda")
    want = qh.qmatmul(w, src)
    big = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    stream, ws = torch.cuda.Stream(), qh.Workspace()
    with torch.cuda.stream(stream):
        x = torch.zeros(8, k, device="cuda")
        for _ in range(8):
            big = big @ big * 1e-3   # some milliseconds of work
        x.copy_(src)
        y = qh.qmatmul(w, x, workspace=ws)
        ys = qh.qmatmul_multi([w, w], x, workspace=ws)
        g = qh.qmatmul_grouped([w], x, None, np.array([0, 8], np.int32), workspace=ws)
        d = w.dequantize()
    stream.synchronize()
    assert torch.equal(y, want) and torch.allclose(ys[0], want, rtol=1e-5, atol=1e-6) and torch.allclose(g, want, rtol=1e-5, atol=1e-6)
    assert torch.equal(d, w.dequantize())


def test_a_given_result_and_an_own_workspace(qh):
    w = weight(qh)
    x = torch.ones(2, 3, 512, device="cuda")

    class Own:
        def get(self, nbytes, device):
            return torch.empty(nbytes + 256, dtype=torch.uint8, device=device)
    out = torch.full((2, 3, 64), float("nan"), device="cuda")
    assert qh.qmatmul(w, x, out=out, workspace=Own()) is out
    assert torch.equal(out, qh.qmatmul(w, x))


def test_dequantize_initialises_torch():
    """A program whose first device tensor is a dequantized weight: torch knows afterwards that the device is in use (its
    memory statistics and its check for forked processes ask for that)."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = ("import torch; from candle_amd import qhip; d = qhip.QWeight.zeros(qhip.Q4K, 64, 512).dequantize(); "
            "assert torch.cuda.is_initialized() and torch.cuda.memory_allocated() >= 64 * 512 * 4; print('ok', flush=True)")
    r = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout, r.stderr[-2000:])
