"""The workspace a matmul asks for, on the CPU: a caller who sized one for a number of rows, and cq_qmatmul_static, whose array
has a fixed size, go by it."""
import ctypes as C

import pytest

from candle_amd import qhip

STATIC = 16 << 20   # CQ_STATIC_SCRATCH_BYTES


class Weight(C.Structure):
    """The head of cq_weight (csrc/qhip_internal.h), all that the size is computed from."""
    _fields_ = [("dev", C.c_int), ("dtype", C.c_int), ("ggml_dtype", C.c_int), ("n", C.c_int64), ("k", C.c_int64),
                ("rest", C.c_uint8 * 256)]


def up(v):
    return (v + 255) // 256 * 256


def bound(k, m):
    """Rows of int8, their scales and block sums in 32 bits each and half of that once more, padded as the kernels read them."""
    pad = (m + 31) // 32 * 32 if m <= 32 else (m + 127) // 128 * 128
    blocks = k // 32
    return up(pad * k) + up(pad * blocks * 4) + up(m * blocks * 4) + up(pad * blocks * 2)


def bytes_of(dtype, k, m, flags=0):
    w = Weight(0, dtype, dtype, 64, k)
    return qhip.load().cq_workspace_bytes(C.byref(w), m, flags)


@pytest.mark.parametrize("dtype,flags", [(qhip.Q8_0, 0), (qhip.Q4_0, 0), (qhip.Q4K, qhip.FLAG_ACT_Q8_1)])
@pytest.mark.parametrize("k", [32, 64, 96, 224, 256, 320, 3200, 4096, 11008, 14336])
def test_rows_of_32_element_blocks(dtype, flags, k):
    if dtype == qhip.Q4K and k % 256:
        pytest.skip("rows of whole 256-element blocks")
    for m in [*range(1, 300), 511, 512, 805, 833, 850, 1003, 1024, 1025, 4096]:
        assert bytes_of(dtype, k, m, flags) <= bound(k, m), (k, m)


@pytest.mark.parametrize("dtype", [qhip.Q8_0, qhip.Q4_0])
def test_most_rows_of_the_static_array(dtype):
    """14336 elements: 850 rows fit the array."""
    assert bytes_of(dtype, 14336, 850) <= STATIC
