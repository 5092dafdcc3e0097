"""The offset terms of Q4_1 / Q5_1 / Q2K by themselves: weights whose blocks (Q2K: groups) are constant have no other part, so that y is the term.
Against the same sum in 64 bits over the values that the kernels read; rows and weight rows of no whole tile, block counts of no whole step and
of fewer steps than the waves that share a tile."""
import numpy as np
import pytest
import torch

from candle_amd.quantized import GgmlDType, QTensor
from oracle import cpu_oracle as orc
from tests.test_gpu_fused_neighbours import qh  # noqa: F401

pytestmark = pytest.mark.gpu

SHAPES = [(1, 40, 64), (6, 100, 11008), (16, 4112, 4096), (4, 100, 4160), (5, 100, 64), (5, 33, 4160), (31, 1000, 576), (33, 70, 1088), (64, 4096, 2112), (65, 16390, 128), (700, 8200, 1088)]


def f16(x):
    return x.astype(np.float16).astype(np.float32)


def rows(m, k, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[m // 2] *= 1e-6        # s in the subnormal f16
    x[m - 1, :32] = 0.0
    return rng, x


def check(y, ref, mag, terms):
    # one f32 rounding for each of the additions (and one of the sum into y), relative to the sum of magnitudes
    assert np.all(np.abs(y - ref) <= (terms + 2) * 2.0**-24 * mag + 1e-30)


@pytest.mark.parametrize("dt", ["Q4_1", "Q5_1"])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_min32(qh, dt, m, n, k):  # noqa: F811
    rng, x = rows(m, k, m + n)
    mins = f16(rng.standard_normal((n, k // 32)) * 0.05)
    w = QTensor.quantize(torch.from_numpy(np.repeat(mins, 32, axis=1)).cuda(), GgmlDType[dt]).weight
    y = torch.full((m + 1, n), 7.0, device="cuda")
    qh.qmatmul(w, torch.from_numpy(x).cuda(), out=y[:m])
    assert bool((y[m] == 7.0).all())
    b = x.reshape(m, k // 32, 32)
    d = np.abs(b).max(axis=2) / np.float32(127.0)
    with np.errstate(divide="ignore", invalid="ignore"):
        t = np.where(d[..., None] != 0, b * (np.float32(1.0) / d)[..., None], np.float32(0.0)).astype(np.float32)
    q = np.trunc(t + np.copysign(np.float32(0.5), t)).astype(np.int32)   # half away from zero
    q = np.where(np.abs(t - np.trunc(t)) < 0.5, np.trunc(t), q).astype(np.int32)
    s = f16(f16(q.sum(axis=2).astype(np.float32)) * f16(d)).astype(np.float64)
    check(y[:m].cpu().numpy(), s @ mins.astype(np.float64).T, np.abs(s) @ np.abs(mins.astype(np.float64)).T, k // 32)


@pytest.mark.parametrize("m,n,k", [(m, n, (k + 255) // 256 * 256) for m, n, k in SHAPES])
def test_min16(qh, m, n, k):  # noqa: F811
    rng, x = rows(m, k, m + n)
    blocks = np.zeros((n, k // 256, 84), dtype=np.uint8)   # scales 0 and minima in the high nibbles, quants 0, d, dmin
    mins = rng.integers(0, 16, (n, k // 256, 16)).astype(np.uint8)
    dmin = (rng.standard_normal((n, k // 256)) * 0.05).astype(np.float16)
    blocks[..., :16] = mins << 4
    blocks[..., 80:82] = np.array([1.0], dtype=np.float16).view(np.uint8)
    blocks[..., 82:] = dmin[..., None].view(np.uint8)
    w = qh.QWeight.from_ggml(orc.Q2K, blocks.reshape(-1), n, k)
    y = torch.full((m + 1, n), 7.0, device="cuda")
    qh.qmatmul(w, torch.from_numpy(x).cuda(), out=y[:m])
    assert bool((y[m] == 7.0).all())
    a = np.concatenate([orc.quantize(orc.Q8K, x[r]) for r in range(m)]).view(np.uint8).reshape(m, k // 256, 292)
    d = np.ascontiguousarray(a[..., :4]).view(np.float32)[..., 0].astype(np.float64)
    sums = np.ascontiguousarray(a[..., 260:]).view(np.int16).astype(np.float64)
    s = (sums * d[..., None]).reshape(m, k // 16)
    v = (mins * dmin.astype(np.float64)[..., None]).reshape(n, k // 16)
    # (two more roundings a block: dmin * d8, and its product with the integer)
    check(y[:m].cpu().numpy(), -(s @ v.T), np.abs(s) @ np.abs(v).T, k // 256 + 2)
