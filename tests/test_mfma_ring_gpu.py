"""The MFMA GEMM kernel's LDS ring at its edges: tile fringes, stages short of
their k, fewer stages than ring slots, 16-byte and 4-byte loads (odd extents,
odd leading dimensions, bases off a 16-byte boundary), leading dimensions past
32-bit offsets.  Bit for bit against the oracle's jmul! recurrence, which both
the FP64 and the FP32 MFMA chains are, signed zeros and denormals included."""
import numpy as np
import pytest

import jblas_amd as jb
from jblas_amd import generators as G
from oracle import oracle as O

from conftest import to_host

pytestmark = pytest.mark.gpu

# around each tile (32, 64, 128), each stage (16, 32 k) and the ring's two to four slots
SHAPES = [(1, 1, 1), (2, 3, 4), (31, 33, 15), (32, 64, 16), (33, 31, 17), (64, 32, 32), (65, 63, 33), (128, 128, 48),
          (127, 130, 64), (129, 127, 65), (200, 66, 100), (140, 260, 129)]


def bits(x):
    return x.view(np.int64 if x.dtype == np.float64 else np.int32)


def special(a, seed):
    """Signed zeros and denormals sprinkled over a."""
    r = np.random.default_rng(seed)
    tiny = np.finfo(a.dtype).tiny
    for v in (0.0, -0.0, tiny / 8, -tiny / 8):
        a[r.random(a.shape) < 0.05] = v
    return a


def placed(torch, a, pad, shift):
    """a on the device, column-major with leading dimension rows + pad, its base `shift` elements off an aligned one."""
    rows, cols = a.shape
    ld = rows + pad
    buf = torch.full((shift + ld * cols,), float("nan"), dtype=torch.float64 if a.dtype == np.float64 else torch.float32,
                     device="cuda")
    v = buf[shift:].view(cols, ld).T[:rows]
    v.copy_(torch.from_numpy(np.ascontiguousarray(a)))
    return v


@pytest.mark.parametrize("tile", ["128", "64", "64x32", "32", ""])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_ring_edges(gpu, dtype, tile, monkeypatch):
    if tile:
        monkeypatch.setenv("JB_GEMM_TILE", tile)
    for si, (m, n, k) in enumerate(SHAPES):
        A = special(G.matrix(70 + si, m, k, dtype=dtype), si)
        X = special(G.matrix(90 + si, k, n, dtype=dtype), 50 + si)
        ref = O.jmul(A, X)
        for ta in "NT":
            for tb in "NT":
                a, x = (A if ta == "N" else A.T), (X if tb == "N" else X.T)
                for pad, shift in ((0, 0), (4, 0), (1, 0), (4, 1)):
                    D = placed(gpu, np.full((m, n), np.nan, dtype=dtype), pad, shift)
                    jb.gemm_(ta, tb, 1.0, placed(gpu, a, pad, shift), placed(gpu, x, pad, shift), 0.0, D)
                    gpu.cuda.synchronize()
                    assert np.array_equal(bits(to_host(D)), bits(ref)), (m, n, k, ta, tb, pad, shift)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("ta,tb", [("T", "N"), ("N", "T")])
def test_ring_wide_leading_dimension(gpu, dtype, ta, tb):
    """Leading dimensions whose stage offsets do not fit 32 bits."""
    m, n, k = 37, 33, 35
    A, X = G.matrix(7, m, k, dtype=dtype), G.matrix(8, k, n, dtype=dtype)
    ld = (1 << 32) // ((128 if ta == "T" else 32) * np.dtype(dtype).itemsize) + 6
    tt = gpu.float64 if dtype == np.float64 else gpu.float32

    def far(a):
        v = gpu.empty(ld * a.shape[1], dtype=tt, device="cuda").view(a.shape[1], ld).T[:a.shape[0]]
        v.copy_(gpu.from_numpy(np.ascontiguousarray(a)))
        return v

    D = jb.device_matrix(m, n, tt)
    jb.gemm_(ta, tb, 1.0, far(A if ta == "N" else A.T), far(X if tb == "N" else X.T), 0.0, D)
    gpu.cuda.synchronize()
    assert np.array_equal(bits(to_host(D)), bits(O.jmul(A, X)))
