"""K-quants with 17 to 32 rows, by the split-K kernel or the tiles (24 rows, short and long weight rows, few and many of them), ragged counts too: a
row's result against the oracle on a part of the weight rows, and the kernel that the rule names."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import cpu_oracle as orc  # noqa: E402
from test_gpu_fused_neighbours import qh  # noqa: E402,F401


@pytest.mark.parametrize("dt", [orc.Q4K, orc.Q5K, orc.Q6K])
@pytest.mark.parametrize("m,k,n", [(17, 1024, 15361), (24, 2048, 16384), (24, 2048, 24576), (25, 2048, 12288), (25, 512, 12300), (32, 8192, 11008),
                                   (32, 14336, 4160)])
def test_either_side_of_the_line(qh, dt, m, k, n):  # noqa: F811
    g = torch.Generator(device="cuda").manual_seed(n + m)
    w = qh.QWeight.zeros(dt, n, k).quantize_(torch.randn(n, k, generator=g, device="cuda") * 0.02)
    x = torch.randn(m, k, generator=g, device="cuda")
    y = qh.qmatmul(w, x).cpu().numpy()
    rows = np.unique(np.r_[0:40, n // 2:n // 2 + 40, n - 40:n])
    row_bytes = k // 256 * orc.TYPE_SIZE[dt]
    want = orc.matmul(dt, x.cpu().numpy(), w.to_ggml().reshape(n, row_bytes)[rows].ravel(), len(rows))
    err = np.linalg.norm(y[:, rows] - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() <= 4 * (k // 256) * 2.0 ** -24 + 1e-6, err.max()   # one f32 addition a block, any order, and the row sums of the blocks


@pytest.mark.parametrize("dt", [orc.Q4K, orc.Q5K, orc.Q6K])
@pytest.mark.parametrize("m,k,n", [(17, 1024, 16384), (24, 2048, 24576), (24, 14336, 8192), (24, 12288, 4096), (24, 12288, 4112), (25, 2048, 12288),
                                   (32, 8192, 11008), (32, 14336, 4160), (32, 3072, 12288), (32, 7168, 2048)])
@pytest.mark.parametrize("det", [False, True])
def test_the_kernel_that_the_rule_names(qh, dt, m, k, n, det):  # noqa: F811
    """The split-K kernel has the same bits wherever it runs and the tiles have others; a deterministic call asks for tiles without K split."""
    g = torch.Generator(device="cuda").manual_seed(n + m)
    w = qh.QWeight.zeros(dt, n, k).quantize_(torch.randn(n, k, generator=g, device="cuda") * 0.02)
    x = torch.randn(m, k, generator=g, device="cuda")
    y, split = qh.qmatmul(w, x, qh.FLAG_DETERMINISTIC if det else 0), qh.qmatmul(w, x, qh.FLAG_FORCE_SKINNY)
    ahead = qh.load()._Z19cq_skinny_few_aheadPK9cq_weightl
    ahead.restype, ahead.argtypes = C.c_bool, [C.c_void_p, C.c_int64]
    if not det:
        assert torch.equal(y, split) == ahead(w.handle, m)
    else:
        assert torch.equal(y, qh.qmatmul(w, x, qh.FLAG_DETERMINISTIC))
        assert not ahead(w.handle, m) or torch.equal(y, split)   # without the split the tiles are no faster
    assert ((y - split).norm() / split.norm()).item() <= 4 * (k // 256) * 2.0 ** -24 + 1e-6
