"""rms_norm quantizer, a row over several workgroups: chunk counts around a workgroup's four and the sixteen that are summed at
a time, ragged last chunks, row counts on both sides of the change to one workgroup per row.  Byte-exact against the same
arithmetic in numpy."""
import numpy as np
import pytest

from oracle import cpu_oracle as orc
from tests.test_gpu_fused_neighbours import canonical_rms_blocks, dev, qh, rms_inputs  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act,m,k", [(orc.Q8K, 1, 2304), (orc.Q8K, 3, 256 * 13), (orc.Q8K, 64, 4096), (orc.Q8K, 65, 4096),
                                     (orc.Q8K, 2, 256 * 17), (orc.Q8K, 4, 256 * 65), (orc.Q8_0, 3, 2080), (orc.Q8_0, 5, 4096 + 32),
                                     (orc.Q8_0, 51, 5120 - 64), (orc.Q8_0, 52, 5120 - 64), (orc.Q8_1, 7, 256 * 9)])
def test_split_rows_bytes(qh, act, m, k):  # noqa: F811
    x, alpha = rms_inputs(k + m, m, k)
    got = qh.quantize_act(act, dev(x), qh.PRE_RMS_NORM, dev(alpha), 1e-5).cpu().numpy()
    assert np.array_equal(got, canonical_rms_blocks(act, x, alpha, 1e-5))


@pytest.mark.parametrize("bad", [np.nan, np.inf, 1e30])
def test_split_row_without_a_finite_scale(qh, bad):  # noqa: F811
    x, alpha = rms_inputs(5, 3, 4096)
    ref = qh.quantize_act(orc.Q8K, dev(x), qh.PRE_RMS_NORM, dev(alpha), 1e-5).cpu().numpy().reshape(3, -1)
    x[1, 3001] = bad
    got = qh.quantize_act(orc.Q8K, dev(x), qh.PRE_RMS_NORM, dev(alpha), 1e-5).cpu().numpy().reshape(3, -1)
    assert not got[1].any()
    assert np.array_equal(got[[0, 2]], ref[[0, 2]])
