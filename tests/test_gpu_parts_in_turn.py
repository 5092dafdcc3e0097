"""K split in two over workgroups (K-quant tile launches, plain and grouped): the two parts of a tile take turns at its results.  Every form of the
launch (one row tile, several of 32, tiles of 64 and of 128 rows; that a call took it is seen in the counters it leaves), rows and weight rows of no
whole tile, an odd number of blocks, outputs that hold NaN before the call, replays of a captured call, calls that reuse the rows (they only read
the workspace, which several streams may then do at once).  Against the launch that does not split (the same block integers, f32 sums over a row's blocks in another
order); from call to call the same bits."""
import numpy as np
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_few_rows_long import close
from tests.test_gpu_fused_neighbours import qh  # noqa: F401

pytestmark = pytest.mark.gpu

# type, weight rows, K, rows, height of the tiles / 32 in the plan for 256 compute units (Q2K and Q3K are held as Q6K)
SHAPES = [("Q4K", 2080, 6144, 1003, 4), ("Q5K", 2081, 4096, 1003, 4), ("Q6K", 3102, 9216, 1089, 4), ("Q3K", 6966, 5632, 280, 4), ("Q2K", 3102, 9216, 1089, 4),
          ("Q6K", 21822, 5376, 97, 4), ("Q4K", 65626, 3072, 33, 2), ("Q5K", 65626, 2560, 33, 2), ("Q6K", 65626, 2048, 33, 2),
          ("Q4K", 704, 2048, 65, 1), ("Q5K", 704, 2816, 45, 1), ("Q6K", 736, 3840, 88, 1)]
ONE_TILE = [("Q4K", 768, 3584, 24, 1), ("Q5K", 800, 3840, 19, 1), ("Q6K", 1600, 3840, 18, 1), ("Q4K", 576, 2048, 10, 1), ("Q5K", 608, 2048, 12, 1),
            ("Q6K", 640, 2304, 16, 1)]


def inputs(dt, n, k, m):
    g = torch.Generator(device="cuda").manual_seed(n + k + m)
    return QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02, GgmlDType[dt]).weight, torch.randn(m, k, generator=g, device="cuda")


def marked_workspace(qh):  # noqa: F811
    ws = qh.Workspace()
    ws.get(64 << 20, torch.device("cuda", 0)).fill_(0xEE)
    return ws


def turns_taken(ws, m, k):
    """The counters of the parts, in the padding rows behind m quantized rows of a marked workspace: how many pairs {turns taken, turns done} both parts of a
    tile and wave have left, and whether none was touched."""
    words = ws.buf[((m + 63) // 64 * 64 + 192) * k:][:64 * k].view(torch.int32).view(-1, 2)
    return int((words == torch.tensor([2, 1], device="cuda", dtype=torch.int32)).all(1).sum()), bool((words == -0x11111112).all())


@pytest.mark.parametrize("dt,n,k,m,mt", SHAPES + ONE_TILE)
def test_two_parts(qh, dt, n, k, m, mt):  # noqa: F811
    w, x = inputs(dt, n, k, m)
    force = qh.FLAG_FORCE_GEMM if mt == 1 else 0   # (of itself the call may go to another kernel)
    want = qh.qmatmul(w, x, qh.FLAG_DETERMINISTIC | force)
    ws, first = marked_workspace(qh), None
    for flags in (0, 0, qh.FLAG_REUSE_ACT, 0):
        out = torch.full((m + 1, n), float("nan"), device="cuda")
        before = ws.buf.clone() if flags else None
        qh.qmatmul(w, x, flags | force, out=out[:m], workspace=ws)
        assert before is None or torch.equal(before, ws.buf)
        assert turns_taken(ws, m, k)[0] == -(-n // 32) * -(-m // (32 * mt))
        assert bool(torch.isnan(out[m]).all())
        close(out[:m], want, k // 256)
        first = out[:m] if first is None else first
        assert torch.equal(first, out[:m])


@pytest.mark.parametrize("dt,n,k,m,mt", [SHAPES[0], SHAPES[2], SHAPES[3], SHAPES[8], SHAPES[10], ONE_TILE[0]])
def test_replays(qh, dt, n, k, m, mt):  # noqa: F811
    w, x = inputs(dt, n, k, m)
    ws = marked_workspace(qh)
    force = qh.FLAG_FORCE_GEMM if mt == 1 else 0   # (of itself the call may go to another kernel)
    qh.qmatmul(w, x, force, workspace=ws)
    y = torch.empty(m, n, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        qh.qmatmul(w, x, force, out=y, workspace=ws)
    for i in range(4):
        x.normal_()
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert turns_taken(ws, m, k)[0] == -(-n // 32) * -(-m // (32 * mt))
        assert torch.equal(y, qh.qmatmul(w, x, force))


# (in five parts: no turns)
@pytest.mark.parametrize("dt,n,k,counts,mt,parts", [
    ("Q4K", 960, 1280, (10, 11, 9, 14, 8, 12, 10, 10), 1, 2), ("Q4K", 2176, 2048, (25, 30, 20, 26, 31, 17, 28, 24), 1, 2),
    ("Q4K", 3648, 5376, (64, 60, 50, 63, 57, 64, 58, 54), 2, 2), ("Q4K", 3200, 6656, (100, 90, 80, 70, 85, 75, 100, 84), 4, 2),
    ("Q5K", 1217, 1280, (10, 11, 9, 14, 8, 12, 10, 10), 1, 2), ("Q5K", 3360, 3072, (64, 60, 50, 63, 57, 64, 58, 52), 2, 2),
    ("Q5K", 3041, 3584, (70, 60, 80, 70, 65, 75, 70, 60), 4, 2), ("Q6K", 4096, 14336, (16, 9, 22, 0, 31, 17, 20, 13), 1, 2),
    ("Q6K", 1216, 1024, (25, 30, 20, 26, 31, 17, 28, 29), 1, 2), ("Q6K", 3552, 4096, (64, 50, 60, 33, 47, 56, 60, 60), 2, 2),
    ("Q6K", 3105, 3584, (70, 60, 80, 70, 65, 35, 70, 60), 4, 2), ("Q4K", 1030, 3584, (40, 25, 1, 33, 20, 30, 26, 25), 1, 5)])
def test_experts(qh, dt, n, k, counts, mt, parts):  # noqa: F811
    """Turns, but for outputs of middle size that the quantizer clears on its way, which are added to (with row ids a launch would have to clear them), and
    for reused rows."""
    experts = [inputs(dt, n, k, 8 + e)[0] for e in range(len(counts))]
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    m = int(offsets[-1])
    x = torch.randn(m, k, device="cuda")
    ids = torch.arange(m, device="cuda", dtype=torch.int32).flip(0).contiguous()
    for rows in (None, ids):
        want = qh.qmatmul_grouped(experts, x, rows, offsets, flags=qh.FLAG_DETERMINISTIC | qh.FLAG_FORCE_GEMM)
        ws = marked_workspace(qh)
        first = qh.qmatmul_grouped(experts, x, rows, offsets, flags=qh.FLAG_FORCE_GEMM, workspace=ws)
        close(first, want, k // 256)
        taken, untouched = turns_taken(ws, m, k)
        if parts == 2 and (rows is not None or not 7 << 15 <= m * n < 7 << 17):
            assert taken == -(-n // 32) * sum(-(-c // (32 * mt)) for c in counts)
        else:
            assert untouched
        for flags in (0, qh.FLAG_REUSE_ACT):
            before = ws.buf.clone()
            again = qh.qmatmul_grouped(experts, x, rows, offsets, flags=qh.FLAG_FORCE_GEMM | flags, workspace=ws)
            assert torch.equal(before, ws.buf)
            close(again, want, k // 256)
            assert parts != 2 or torch.equal(first, again)   # (a sum of two has the same bits in either order)


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
