"""The choices of a kernel by sizes, on the CPU: measured shapes (us, whole calls, weights from HBM) where one kernel is clearly ahead get that one."""
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


def rule(mangled, w, m):
    """A function bool(const cq_weight *, int64_t) of the library's insides."""
    f = getattr(qhip.load(), mangled)
    f.restype, f.argtypes = C.c_bool, [C.c_void_p, C.c_int64]
    return f(w, m)


def weight(dt, n, k):
    held = {qhip.Q4_1: qhip.Q8_0, qhip.Q5_1: qhip.Q8_0, qhip.Q2K: qhip.Q6K}   # whose planes they are stored as
    return Weight(0, held.get(dt, dt), dt, n, k)


@pytest.mark.parametrize("dt,n,k,m,split,tiles", FASTER)
def test_split_k_or_tiles(dt, n, k, m, split, tiles):
    """17 to 32 rows of a K-quant."""
    w = weight(dt, n, k)
    assert rule("_Z19cq_skinny_few_aheadPK9cq_weightl", C.addressof(w), m) == (split < tiles)


@pytest.mark.parametrize("dt,n,k,m,one,split", [
    (qhip.Q2K, 32000, 2048, 2, 19.9, 21.2), (qhip.Q2K, 32000, 2048, 4, 28.7, 21.1),
    (qhip.Q2K, 8192, 1024, 2, 6.9, 7.3), (qhip.Q2K, 8192, 1024, 4, 10.1, 7.5), (qhip.Q2K, 4096, 11008, 2, 24.3, 15.7), (qhip.Q2K, 1024, 12288, 2, 13.7, 14.2),
    (qhip.Q4_1, 32000, 1024, 2, 14.7, 16.0), (qhip.Q4_1, 32000, 1024, 4, 20.1, 16.5), (qhip.Q4_1, 32000, 4096, 3, 34.3, 37.7)])
def test_one_launch_or_split_k_for_the_offset_types(dt, n, k, m, one, split):
    """Two to four rows; the one launch, whose rows have the bits of their one-row calls, is favoured by 12 %."""
    w = weight(dt, n, k)
    assert rule("_Z30cq_matvec_fused_rows_supportedPK9cq_weightl", C.addressof(w), m) == (one < 1.12 * split)


@pytest.mark.parametrize("dt,n,k,m,two,one", [
    (qhip.Q4K, 4096, 4096, 2, 9.1, 6.0), (qhip.Q4K, 4096, 4096, 4, 9.3, 8.7), (qhip.Q4K, 32000, 4096, 2, 26.8, 22.6), (qhip.Q4K, 32000, 4096, 4, 26.3, 28.0),
    (qhip.Q6K, 32000, 2048, 2, 19.8, 18.4), (qhip.Q6K, 32000, 2048, 3, 20.6, 22.4), (qhip.Q5K, 4096, 4096, 3, 10.5, 7.8)])
def test_rms_norm_in_the_one_launch_or_in_front(dt, n, k, m, two, one):
    """Two to four rows behind rms_norm: the quantizer and the kernel behind it, or one launch."""
    w = weight(dt, n, k)
    ws = (C.c_void_p * 1)(C.addressof(w))
    f = qhip.load()._Z34cq_matvec_fused_rms_rows_supportedPKPK9cq_weightil
    f.restype, f.argtypes = C.c_bool, [C.c_void_p, C.c_int, C.c_int64]
    assert f(ws, 1, m) == (one < two)
