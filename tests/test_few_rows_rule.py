"""The choice between the split-K kernel and the tiles for 17 to 32 rows of a K-quant, on the CPU: measured shapes (us, split K / tiles, whole calls,
weights from HBM) where one of them is clearly ahead get that one."""
import ctypes as C

import pytest

from candle_amd import qhip
from test_workspace_bytes import Weight

FASTER = [   # dtype, weight rows, K, rows, split K, tiles
    (qhip.Q4K, 8192, 14336, 17, 32.0, 25.8), (qhip.Q4K, 8192, 14336, 24, 31.8, 26.6), (qhip.Q4K, 4128, 12288, 24, 25.6, 19.8),
    (qhip.Q4K, 4096, 11008, 24, 16.0, 18.3), (qhip.Q4K, 4096, 14336, 24, 18.9, 21.0), (qhip.Q4K, 32000, 4096, 24, 33.4, 29.6),
    (qhip.Q5K, 14336, 2048, 24, 15.9, 18.4), (qhip.Q5K, 16384, 3072, 24, 19.7, 23.8), (qhip.Q5K, 6144, 16384, 24, 38.3, 33.7),
    (qhip.Q6K, 12288, 3072, 24, 16.5, 22.9), (qhip.Q6K, 4096, 14336, 24, 21.9, 26.7), (qhip.Q4K, 11008, 8192, 32, 32.5, 25.5),
    (qhip.Q4K, 10240, 1024, 32, 11.6, 9.9), (qhip.Q4K, 4096, 14336, 32, 20.8, 22.0), (qhip.Q6K, 8192, 14336, 32, 41.1, 34.7),
    (qhip.Q6K, 12288, 3072, 32, 20.3, 23.4), (qhip.Q4K, 128256, 512, 32, 72.7, 22.6)]


@pytest.mark.parametrize("dt,n,k,m,split,tiles", FASTER)
def test_the_faster_kernel_is_taken(dt, n, k, m, split, tiles):
    ahead = qhip.load()._Z19cq_skinny_few_aheadPK9cq_weightl   # cq_skinny_few_ahead(const cq_weight *, int64_t)
    ahead.restype, ahead.argtypes = C.c_bool, [C.c_void_p, C.c_int64]
    w = Weight(0, dt, dt, n, k)
    assert ahead(C.addressof(w), m) == (split < tiles)
