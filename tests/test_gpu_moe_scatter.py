"""The two ways the experts' rows go back to their tokens: added to what the destination holds, and written whatever it holds; both kernels (rows of a
multiple of four elements or not, destinations off sixteen bytes), tokens without a row, no rows at all.  Bit for bit the sequential sums."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from test_gpu_fused_neighbours import qh  # noqa: E402,F401


@pytest.mark.parametrize("tokens,total,hidden,off", [(5, 9, 6, 0), (7, 130, 8, 0), (3, 70, 1028, 0), (3, 70, 1028, 1), (4, 0, 16, 0), (4, 0, 5, 0)])
def test_added_and_written(qh, tokens, total, hidden, off):  # noqa: F811
    rng = np.random.default_rng(tokens + total + off)
    y = rng.standard_normal((total, hidden)).astype(np.float32)
    rid = rng.integers(0, tokens - 1, size=total).astype(np.int32)   # the last token gets no row
    wt = rng.random(total).astype(np.float32)
    held = rng.standard_normal((tokens, hidden)).astype(np.float32)
    y_d, rid_d, wt_d = (torch.from_numpy(v).cuda() for v in (y, rid, wt))
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for entry, start in (("cq_moe_scatter_add", held), ("cq_moe_scatter", np.zeros_like(held))):
        want = start.copy()
        for p in range(total):
            want[rid[p]] = want[rid[p]] + y[p] * wt[p]
        buf = torch.full((tokens * hidden + off + 1,), float("nan"), device="cuda")
        ys = buf[off:-1].view(tokens, hidden)
        if entry == "cq_moe_scatter_add":
            ys.copy_(torch.from_numpy(held))
        qh.check(getattr(qh.load(), entry)(0, y_d.data_ptr(), rid_d.data_ptr(), wt_d.data_ptr(), total, hidden, ys.data_ptr(), tokens, stream))
        assert np.array_equal(ys.cpu().numpy().view(np.uint32), want.view(np.uint32))
        assert bool(torch.isnan(buf[-1]))
