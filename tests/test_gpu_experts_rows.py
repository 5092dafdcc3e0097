"""Grouped calls with more rows an expert than a tile of the split-K kernel holds, and the choice between it and the tile kernels: experts without
rows, with one, at the edges of 8, 16, 24 and 32 rows, weight rows of no whole tile.  Against a call of each expert's rows by itself on the
dot-product kernel of the staged path: the same block integers, f32 sums over a row's blocks in another order."""
import numpy as np
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from tests.test_gpu_fused_neighbours import qh  # noqa: F401
from tests.test_gpu_few_rows_long import close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["Q4K", "Q5K", "Q6K", "Q3K", "Q8_0", "Q4_0", "Q5_0"])
@pytest.mark.parametrize("n,k,rows", [(130, 512, (0, 17, 1, 16, 25)), (1792, 1024, (9, 16, 15, 10, 8, 12)), (1030, 768, (24, 23, 33, 0, 32, 8)),
                                      (3072, 2560, (11, 18, 12, 13, 14, 16, 16, 17)), (512, 256, (100, 1, 64, 49)), (40, 1280, (400, 3, 700)),
                                      (33, 256, (1700, 900)), (1536, 4096, (21, 24, 19, 23))])
def test_rows_beyond_a_tile(qh, dt, n, k, rows):  # noqa: F811
    g = torch.Generator(device="cuda").manual_seed(n + k + len(rows))
    ws = [QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02, GgmlDType[dt]).weight for _ in rows]
    off = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    x = torch.randn(int(off[-1]), k, generator=g, device="cuda")
    want = torch.cat([qh.qmatmul(w, x[a:b].contiguous(), qh.FLAG_FORCE_MATVEC | qh.FLAG_STAGED_ACT) for w, a, b in zip(ws, off, off[1:]) if b > a])
    blocks = k // (256 if dt.endswith("K") else 32)
    close(qh.qmatmul_grouped(ws, x, None, off), want, blocks)
    close(qh.qmatmul_grouped(ws, x, None, off, flags=qh.FLAG_FORCE_SKINNY), want, blocks)
    bad = x.clone()
    bad[off[-1] - 1, 3], bad[0, k - 1] = float("inf"), float("nan")
    same = [qh.qmatmul_grouped(ws, v, None, off, flags=qh.FLAG_DETERMINISTIC)[1:-1] for v in (bad, x)]
    assert torch.equal(*same)


@pytest.mark.parametrize("dt", ["Q4K", "Q5K", "Q6K", "Q8_0", "Q4_0"])
@pytest.mark.parametrize("n,k,rows", [(256, 2304, (33, 70, 65)), (300, 1536, (20, 31, 5)), (512, 8448, (1, 40)), (64, 512, (130, 0, 129)),
                                      (2048, 1792, (40, 60, 90, 33)), (8200, 512, (700, 1000, 900))])
def test_parts_of_k_and_tile_heights(qh, dt, n, k, rows):  # noqa: F811
    """The tile kernels with parts of two blocks and more, equal or not, added up by one, two and four row tiles a workgroup."""
    g = torch.Generator(device="cuda").manual_seed(n + k)
    ws = [QTensor.quantize(torch.randn(n, k, generator=g, device="cuda") * 0.02, GgmlDType[dt]).weight for _ in rows]
    off = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    x = torch.randn(int(off[-1]), k, generator=g, device="cuda")
    want = torch.cat([qh.qmatmul(w, x[a:b].contiguous(), qh.FLAG_FORCE_MATVEC | qh.FLAG_STAGED_ACT) for w, a, b in zip(ws, off, off[1:]) if b > a])
    blocks = k // (256 if dt.endswith("K") else 32)
    close(qh.qmatmul_grouped(ws, x, None, off, flags=qh.FLAG_FORCE_GEMM), want, blocks)
    close(qh.qmatmul_grouped(ws, x, None, off, flags=qh.FLAG_FORCE_GEMM | qh.FLAG_DETERMINISTIC), want, blocks)


@pytest.mark.parametrize("dt", ["Q8_0", "Q4_0"])
@pytest.mark.parametrize("n,k,rows", [(256, 2112, (33, 20, 32)), (300, 576, (40, 64, 5)), (4100, 320, (300, 128, 129)), (8200, 320, (700, 1000, 900))])
def test_steps_of_no_whole_length(qh, dt, n, k, rows):  # noqa: F811
    test_parts_of_k_and_tile_heights(qh, dt, n, k, rows)
