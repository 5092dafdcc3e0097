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
