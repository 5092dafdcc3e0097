"""Mixture-of-experts projections with few rows per expert: the grouped split-K launch (every row-group count, tiles that
start at any row, empty experts) and the grouped tile launch of the 32-element-block types, against one matmul per expert."""
import numpy as np
import pytest

from oracle import cpu_oracle as orc

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [orc.Q4K, orc.Q5K, orc.Q6K, orc.Q3K, orc.Q8_0, orc.Q4_0, orc.Q5_0])
@pytest.mark.parametrize("rows,k,n", [([1], 256, 16), ([0, 1, 3, 8], 768, 47), ([9, 0, 1], 2304, 130), ([20, 2, 1, 17], 512, 256), ([31, 33, 1], 1024, 100),
                                      ([64, 2, 90], 512, 333), ([130, 40, 257, 70], 256, 4000), ([1, 0, 0, 1, 0, 0, 0, 0], 4096, 96), ([5] * 20, 256, 40)])
def test_against_each_expert(dt, rows, k, n):
    from candle_amd import qhip
    if dt in (orc.Q8_0, orc.Q4_0, orc.Q5_0) and k > 256:
        k -= 64   # a last K step of six blocks
    rng = np.random.default_rng(dt + k + n)
    blocks = [orc.quantize(dt, (rng.standard_normal((n, k)) * 0.03).astype(np.float32)) for _ in rows]
    experts = [qhip.QWeight.from_ggml(dt, b, n, k) for b in blocks]
    offsets = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    x = rng.standard_normal((7, k)).astype(np.float32)
    rid = rng.integers(0, 7, size=int(offsets[-1])).astype(np.int32)
    flags = [0, qhip.FLAG_FORCE_SKINNY, qhip.FLAG_DETERMINISTIC]
    for fl in flags:
        y = qhip.qmatmul_grouped(experts, torch.from_numpy(x).cuda(), torch.from_numpy(rid).cuda(), offsets, flags=fl,
                                 workspace=qhip.Workspace()).cpu().numpy().astype(np.float64)
        for e in range(len(rows)):
            lo, hi = int(offsets[e]), int(offsets[e + 1])
            if lo < hi:
                want = orc.matmul(dt, x[rid[lo:hi]], blocks[e], n)
                assert np.linalg.norm(y[lo:hi] - want) <= 1e-5 * np.linalg.norm(want), (fl, e)
