"""K split in two over workgroups (K-quant tile launches, plain and grouped): the two parts of a tile take turns at its results.  Rows and weight rows of
no whole tile, an odd number of blocks, outputs that hold NaN before the call, replays of a captured call, calls that reuse the rows (they only read
the workspace, which several streams may then do at once).  Against the launch that does not split (the same block integers, f32 sums over a row's blocks in another
order); from call to call the same bits."""
import numpy as np
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_few_rows_long import close
from tests.test_gpu_fused_neighbours import qh  # noqa: F401

pytestmark = pytest.mark.gpu

SHAPES = [("Q4K", 2304, 3584, 1052), ("Q6K", 3102, 9216, 1089), ("Q3K", 6966, 5632, 280), ("Q5K", 2305, 3840, 1040), ("Q2K", 3102, 9216, 1089),
          ("Q6K", 21822, 5376, 97)]


def inputs(dt, n, k, m):
    g = torch.Generator(device="cuda").manual_seed(n + k + m)
    return QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02, GgmlDType[dt]).weight, torch.randn(m, k, generator=g, device="cuda")


@pytest.mark.parametrize("dt,n,k,m", SHAPES)
def test_two_parts(qh, dt, n, k, m):  # noqa: F811
    w, x = inputs(dt, n, k, m)
    want = qh.qmatmul(w, x, qh.FLAG_DETERMINISTIC)
    ws, first = qh.Workspace(), None
    for flags in (0, 0, qh.FLAG_REUSE_ACT, 0):
        out = torch.full((m + 1, n), float("nan"), device="cuda")
        before = ws.buf.clone() if flags else None
        qh.qmatmul(w, x, flags, out=out[:m], workspace=ws)
        assert before is None or torch.equal(before, ws.buf)
        assert bool(torch.isnan(out[m]).all())
        close(out[:m], want, k // 256)
        first = out[:m] if first is None else first
        assert torch.equal(first, out[:m])


@pytest.mark.parametrize("dt,n,k,m", SHAPES[:3])
def test_replays(qh, dt, n, k, m):  # noqa: F811
    w, x = inputs(dt, n, k, m)
    ws = qh.Workspace()
    qh.qmatmul(w, x, workspace=ws)
    y = torch.empty(m, n, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        qh.qmatmul(w, x, out=y, workspace=ws)
    for i in range(4):
        x.normal_()
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, qh.qmatmul(w, x))


@pytest.mark.parametrize("dt,n,k,counts", [("Q6K", 4096, 14336, (16, 9, 22, 0, 31, 17, 20, 13)), ("Q4K", 1030, 3584, (40, 25, 1, 33, 20, 30, 26, 25)),
                                           ("Q5K", 2048, 7168, (10, 12, 8, 9, 14, 6, 11, 10))])
def test_experts(qh, dt, n, k, counts):  # noqa: F811
    experts = [inputs(dt, n, k, 8 + e)[0] for e in range(len(counts))]
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    x = torch.randn(int(offsets[-1]), k, device="cuda")
    ids = torch.arange(x.shape[0], device="cuda", dtype=torch.int32).flip(0).contiguous()
    for rows in (None, ids):
        want = qh.qmatmul_grouped(experts, x, rows, offsets, flags=qh.FLAG_DETERMINISTIC | qh.FLAG_FORCE_GEMM)
        for _ in range(3):
            close(qh.qmatmul_grouped(experts, x, rows, offsets, flags=qh.FLAG_FORCE_GEMM), want, k // 256)
    ws = qh.Workspace()
    want = qh.qmatmul_grouped(experts, x, ids, offsets, flags=qh.FLAG_FORCE_GEMM, workspace=ws)
    before = ws.buf.clone()
    close(qh.qmatmul_grouped(experts, x, ids, offsets, flags=qh.FLAG_FORCE_GEMM | qh.FLAG_REUSE_ACT, workspace=ws), want, k // 256)
    assert torch.equal(before, ws.buf)


def turns_taken(ws, m, k):
    """The counters of the parts in the padding rows of a workspace of m quantized rows that held 0xEE before the call: {turns taken, turns done} of every
    tile and wave that took them."""
    words = ws.buf[((m + 63) // 64 * 64 + 192) * k:][:64 * k].view(torch.int32).view(-1, 2)
    return int((words == torch.tensor([2, 1], device="cuda", dtype=torch.int32)).all(1).sum()), int((words == -0x11111112).all(1).sum()), len(words)


@pytest.mark.parametrize("dt,n,k,counts,by_turns", [("Q4K", 960, 1280, (10, 11, 9, 14, 8, 12, 10, 10), True), ("Q4K", 2176, 2048, (25, 30, 20, 26, 31, 17, 28, 24), False),
                                                    ("Q6K", 1216, 1024, (25, 30, 20, 26, 31, 17, 28, 29), False), ("Q6K", 3552, 4096, (64, 50, 60, 33, 47, 56, 60, 60), True)])
def test_experts_take_turns_where_ahead(qh, dt, n, k, counts, by_turns):  # noqa: F811
    """Outputs of middle size that the quantizer clears are added to; where a launch would have to clear them (row ids) the parts take turns."""
    experts = [inputs(dt, n, k, 8 + e)[0] for e in range(len(counts))]
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    m = int(offsets[-1])
    x = torch.randn(m, k, device="cuda")
    ids = torch.arange(m, device="cuda", dtype=torch.int32)
    want = qh.qmatmul_grouped(experts, x, None, offsets, flags=qh.FLAG_DETERMINISTIC | qh.FLAG_FORCE_GEMM)
    for rows in (None, ids):
        ws = qh.Workspace()
        ws.get(64 << 20, x.device).fill_(0xEE)
        close(qh.qmatmul_grouped(experts, x, rows, offsets, flags=qh.FLAG_FORCE_GEMM, workspace=ws), want, k // 256)
        taken, untouched, pairs = turns_taken(ws, m, k)
        assert taken >= (n + 31) // 32 * len(counts) if by_turns or rows is not None else untouched == pairs


@pytest.mark.parametrize("taken,done,held,want", [(0, 0, float("nan"), 0.0), (1, 1, 0.5, 0.5), (1, 0, 0.5, None), (2, 1, 0.5, None)])
def test_a_turn(qh, taken, done, held, want):  # noqa: F811
    """The first part stores, the second adds; where the first does not come, or there is a third, the results say so."""
    turn = torch.tensor([taken, done], device="cuda", dtype=torch.int32)
    y = torch.full((33, 32), held, device="cuda")
    y[32] = 7.0
    for looks in (0, -1):
        assert qh.load().cq_selfcheck_turns(0, turn.data_ptr(), y.data_ptr(), looks, None) == -1
    torch.cuda.synchronize()
    qh.check(qh.load().cq_selfcheck_turns(0, turn.data_ptr(), y.data_ptr(), 4, torch.cuda.current_stream().cuda_stream))
    assert turn.tolist() == [taken + 1, 1 if taken == 0 else done]
    assert bool((y[32] == 7.0).all())
    if want is None:
        assert bool(torch.isnan(y[:32]).all())
    else:
        assert torch.equal(y[:32], (torch.arange(32, device="cuda") + (1.0 + want)).expand(32, 32))
