"""The grouped 3xBF16 kernels' split into BF16 planes, entry by entry: products with a power
of two on the diagonal bring each entry back alone.

  * Entries whose planes are all normal (2^-100 and up, to the largest finite value): the
    three planes hold all 24 bits, so the product is the entry times the power, exactly.
  * Smaller ones, down to FP32 denormals: bit for bit the product of the single-problem
    kernel, whose split (by subtraction) is kernels of its own.
"""
import numpy as np
import pytest

import jblas_amd as jb
from jblas_amd.grouped import GemmDesc

from conftest import to_dev, to_host
from test_grouped_gpu import write_table

pytestmark = pytest.mark.gpu

ROWS, K = 192, 64
# low halves and low bytes on both sides of the ties of the first and second rounding
LOW = [0, 1, 0x7F, 0x80, 0x81, 0x7FFF, 0x8000, 0x8001, 0xFFFF, 0x17FFF, 0x18000, 0x18001, 0x80FF, 0x7F80, 0x8080, 0x7FFFFF,
       0x7F8000, 0x7F7FFF, 0x7FFF80, 0x7F0080]
NORMAL = [-100, -60, -3, -1, 0, 1, 2, 60, 100, 125, 126, 127]
SMALL = [-126, -125, -120, -118, -112, -110, -109, -103]


def entries(exponent, seed):
    """ROWS x K entries of one binary exponent (None: FP32 denormals), every low part with every sign, signed zeros."""
    r = np.random.default_rng(1000 + seed)
    low = r.integers(0, 1 << 23, ROWS * K).astype(np.uint32)
    low[::3] = np.resize(np.array(LOW, np.uint32), low[::3].size)
    bits = low if exponent is None else low | np.uint32((exponent + 127) << 23)
    bits[5::97] = 0
    return (bits | (r.integers(0, 2, bits.size).astype(np.uint32) << 31)).view(np.float32).reshape(ROWS, K)


def op(a, t):
    return np.asfortranarray(a if t == "N" else a.T)


@pytest.mark.parametrize("cfg", [0, 3, 4, 5])
@pytest.mark.parametrize("side", ["A", "B"])
@pytest.mark.parametrize("t", ["N", "T"])
def test_x3_planes(gpu, cfg, side, t, tmp_path):
    groups = [(e, entries(e, 11 + e), np.float32(2.0 ** min(max(-e, -126), 100))) for e in NORMAL + SMALL]
    groups.append((None, entries(None, 5), np.float32(2.0**120)))
    m, n = (ROWS, K) if side == "A" else (K, ROWS)
    jb.tune_reset()
    write_table(str(tmp_path / "t.json"), "f32_bf16x3", [(m, n, K)], cfg, 1)
    try:
        descs, single = [], []
        for _, x, d in groups:
            diag = np.diag(np.full(K, d, np.float32))
            a, b = (x, diag) if side == "A" else (diag, x.T)
            a, b = to_dev(gpu, op(a, t)), to_dev(gpu, op(b, t))
            descs.append(GemmDesc(t, t, 1.0, a, b, 0.0, jb.device_matrix(m, n, gpu.float32)))
            single.append(jb.gemm_(t, t, 1.0, a, b, 0.0, jb.device_matrix(m, n, gpu.float32), method="bf16x3"))
        jb.gemm_grouped_("f32_bf16x3", descs)
        for (e, x, d), g, s in zip(groups, descs, single):
            got = to_host(g.C) if side == "A" else to_host(g.C).T
            if e in NORMAL:
                assert np.array_equal(got, x * d), e  # (exact in FP32: a power of two)
            else:
                assert np.array_equal(got, to_host(s) if side == "A" else to_host(s).T), e
    finally:
        jb.tune_reset()
