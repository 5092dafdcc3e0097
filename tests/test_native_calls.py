"""The native side of qhip's calls (csrc/calls.cpp) on arguments that never reach a kernel, without a GPU: device tensors are
torch's fake ones, which have no memory, and the C library behind the calls is a handful of Python callbacks.

Each check runs in a process of its own, since what it guards against ends the process."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
N, K = 64, 256


def bind():
    """qhip with its native calls on a stand-in for the C library: every weight is [N, K], every call succeeds."""
    import ctypes as C

    from candle_amd import qhip
    native = qhip._calls()
    vp, i64, ci, sz = C.c_void_p, C.c_int64, C.c_int, C.c_size_t

    def shape(_w, n, k):
        n[0], k[0] = N, K
        return 0
    table = {name: C.CFUNCTYPE(ci)(lambda: 0) for name in qhip.EXPORTS}
    table["cq_weight_shape"] = C.CFUNCTYPE(ci, vp, C.POINTER(i64), C.POINTER(i64))(shape)
    table["cq_workspace_bytes"] = C.CFUNCTYPE(sz, vp, i64, ci)(lambda w, m, f: 256)
    table["cq_grouped_workspace_bytes"] = C.CFUNCTYPE(sz, vp, ci, i64, ci)(lambda w, e, t, f: 256)
    qhip._kept = table
    native.bind({name: C.cast(f, vp).value for name, f in table.items()}, qhip.QHipError, qhip.Workspace)

    class Weight:
        _addr, shape = 1, (N, K)
    return qhip, Weight()


def fake(*shape):
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        return torch.empty(*shape, device="cuda")


def raises(kind, call):
    """The call raises exactly what `kind` names."""
    try:
        call()
    except kind as e:
        print("ok", type(e).__name__, str(e)[:60], flush=True)
    else:
        raise AssertionError("no error")


def child_no_memory():
    """Tensors without memory in each place whose address a call takes (x, the workspace, a given result), plain and behind
    the wrappers of vmap and grad: a Python exception each."""
    import numpy as np
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    qhip, w = bind()
    out, offsets = torch.empty(2, N), np.array([0, 2], np.int32)

    def over(v):   # a workspace whose buffer is the wrapped tensor itself
        ws = qhip.Workspace()
        ws.buf = v
        return ws
    calls = (lambda v: qhip.qmatmul(w, v, out=out), lambda v: qhip.qmatmul(w, v, out=out, pre=qhip.PRE_SILU_MUL, aux=v),
             lambda v: qhip.qmatmul(w, v, out=out, workspace=over(v)), lambda v: qhip.qmatmul_multi([w, w], v, workspace=over(v)),
             lambda v: qhip.qmatmul_grouped([w], v, None, offsets, workspace=over(v)))
    for call in calls:
        with FakeTensorMode():
            x = torch.empty(3, 2, K, device="cuda")
            raises(RuntimeError, lambda: call(x[0]))
            raises(RuntimeError, lambda: torch.func.vmap(call)(x))
            raises(RuntimeError, lambda: torch.func.grad(lambda v: call(v).sum())(x[0]))


def child_second_operand():
    """A second operand that is no tensor is refused with every fused step; without one qmatmul_multi looks at it all the same
    (the other two calls do not read it)."""
    import numpy as np
    qhip, w = bind()
    x, offsets = fake(2, K), np.array([0, 2], np.int32)
    for aux in (1.5, [1.0], "aux", object(), np.ones((2, K), np.float32)):
        for pre in (qhip.PRE_NONE, qhip.PRE_RMS_NORM, qhip.PRE_SILU_MUL, 3):
            bad = (qhip.QHipError, AttributeError)   # (the wording of the refusal asks `aux` whether it is on the device)
            raises(bad, lambda: qhip.qmatmul_multi([w, w], x, pre=pre, aux=aux))
            if pre != qhip.PRE_NONE:
                raises(bad, lambda: qhip.qmatmul(w, x, pre=pre, aux=aux))
                raises(bad, lambda: qhip.qmatmul_grouped([w], x, None, offsets, pre=pre, aux=aux))


def child_many_weights():
    """Any number of weights: 300 of them get as far as one does, to the allocation of the result."""
    import numpy as np
    qhip, w = bind()
    x, ws = fake(2, K), qhip.Workspace()
    ws.buf = fake(1024)
    for count in (1, 256, 257, 300):
        offsets = np.full(count + 1, 2, np.int32)
        offsets[0] = 0
        for call in (lambda: qhip.qmatmul_grouped([w] * count, x, None, offsets, workspace=ws),
                     lambda: qhip.qmatmul_multi([w] * count, x, workspace=ws)):
            try:
                call()
            except RuntimeError as e:
                assert not isinstance(e, qhip.QHipError), (count, e)


def child_gone_weight():
    """A weight that has been given back is refused by every call."""
    import numpy as np
    from candle_amd import qhip   # (on the C library itself)
    w, x = qhip.QWeight(None, 0), fake(2, K)
    for call in (lambda: w.dequantize(), lambda: w.dequantize_f16(), lambda: qhip.qmatmul(w, x), lambda: qhip.qmatmul_multi([w], x),
                 lambda: qhip.qmatmul_grouped([w], x, None, np.array([0, 2], np.int32))):
        raises(qhip.QHipError, call)


def child_other_workspaces():
    """A caller's own workspace is anything with a `get`, and a Workspace's own `get` is asked where a class brings one."""
    import numpy as np
    qhip, w = bind()
    x, buf, offsets = fake(2, K), fake(1024), np.array([0, 2], np.int32)

    class Own:
        asked = 0

        def get(self, nbytes, device):
            self.asked += 1
            return buf

    class Pooled(qhip.Workspace):
        asked = 0
        get = Own.get
    pooled = Pooled()
    pooled.buf = buf
    for ws in (Own(), pooled):
        for call in (lambda: qhip.qmatmul(w, x, workspace=ws), lambda: qhip.qmatmul_multi([w, w], x, workspace=ws),
                     lambda: qhip.qmatmul_grouped([w], x, None, offsets, workspace=ws)):
            raises(RuntimeError, call)   # (the allocation of the result)
        assert ws.asked == 3, ws.asked
    Own.get = lambda self, nbytes, device: 7
    raises(TypeError, lambda: qhip.qmatmul(w, x, workspace=Own()))


def child_eps():
    """`eps` belongs to the fused step: without one nothing reads it."""
    import numpy as np
    qhip, w = bind()
    x, ws, offsets = fake(2, K), qhip.Workspace(), np.array([0, 2], np.int32)
    ws.buf = fake(1024)
    alpha = fake(K)
    for call in (lambda **a: qhip.qmatmul(w, x, workspace=ws, **a), lambda **a: qhip.qmatmul_grouped([w], x, None, offsets, workspace=ws, **a)):
        raises(RuntimeError, lambda: call(eps=None))   # (the allocation of the result)
        raises(TypeError, lambda: call(pre=qhip.PRE_RMS_NORM, aux=alpha, eps=None))


CHILDREN = {f[len("child_"):]: g for f, g in list(globals().items()) if f.startswith("child_")}


@pytest.mark.parametrize("name", CHILDREN)
def test_native_calls(name):
    pytest.importorskip("torch")
    r = subprocess.run([sys.executable, os.path.abspath(__file__), name], cwd=ROOT, capture_output=True, text=True, timeout=300,
                       env={**os.environ, "PYTHONPATH": ROOT, "HIP_VISIBLE_DEVICES": "-1"})
    assert r.returncode == 0, (r.returncode, r.stdout[-1500:], r.stderr[-3000:])


def test_the_weight_is_the_tensor_of_the_call(monkeypatch):
    """QMatMul reads its tensor when it is called: a tensor put in its place is the one that is used, by every form."""
    pytest.importorskip("torch")
    from candle_amd import qhip
    from candle_amd.quantized import QMatMul

    class Tensor:
        def __init__(self, weight):
            self.weight = weight

        def rank(self):
            return 2
    monkeypatch.setattr(qhip, "qmatmul", lambda w, *a, **kw: w)
    monkeypatch.setattr(qhip, "qmatmul_multi", lambda ws, *a, **kw: ws)
    mat = QMatMul(Tensor("first"))
    assert mat.forward(None) == "first"
    mat.qtensor = Tensor("second")
    assert [mat.forward(None), mat.forward_rms_norm(None, None, 0.0), mat.forward_silu_mul(None, None)] == ["second"] * 3
    assert QMatMul.forward_multi([mat, mat], None) == ["second"] * 2


if __name__ == "__main__":
    CHILDREN[sys.argv[1]]()
