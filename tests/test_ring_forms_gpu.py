"""Forms of operands the ring kernels take that the edge tests leave out, bit for bit against
the oracle's recurrence: Float32 operands with Inf, NaN and overflowing products, and leading
dimensions past 32-bit offsets in every transpose combination, single and grouped."""
import numpy as np
import pytest

import jblas_amd as jb
from jblas_amd import generators as G
from jblas_amd.grouped import GemmDesc
from oracle import oracle as O

from conftest import to_dev, to_host
from test_grouped_gpu import write_table

pytestmark = pytest.mark.gpu


def bits(x):
    return np.ascontiguousarray(x).view(np.int64 if x.dtype == np.float64 else np.int32)


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
def test_f32_nonfinite_matches_recurrence(gpu, ta, tb, monkeypatch):
    m, n, k = 150, 90, 120
    A, B = G.matrix(71, m, k, dtype=np.float32), G.matrix(72, k, n, dtype=np.float32)
    A[3, 7], A[40, 0], A[149, 119] = np.inf, -np.inf, np.nan
    B[5, 11], B[119, 89] = np.nan, -np.inf
    A[60, :] *= np.float32(1e38)  # row 60 overflows against B's larger entries
    B[:, 20] *= np.float32(1e10)
    ref = O.jmul(A, B)
    assert np.isinf(ref).sum() > 20 and np.isnan(ref).sum() > n
    nan = np.isnan(ref)
    a, b = to_dev(gpu, A if ta == "N" else A.T), to_dev(gpu, B if tb == "N" else B.T)
    for tile in ("128", "64", "64x32", "32", "jmul", "grouped"):
        C = jb.device_matrix(m, n, gpu.float32)
        if tile == "jmul":
            jb.jmul_(C, to_dev(gpu, A), to_dev(gpu, B))
        elif tile == "grouped":
            jb.gemm_grouped_("f32", [GemmDesc(ta, tb, 1.0, a, b, 0.0, C)])
        else:
            monkeypatch.setenv("JB_GEMM_TILE", tile)
            jb.gemm_(ta, tb, 1.0, a, b, 0.0, C)
            monkeypatch.delenv("JB_GEMM_TILE")
        got = to_host(C)
        assert np.array_equal(np.isnan(got), nan), tile
        assert np.array_equal(bits(got)[~nan], bits(ref)[~nan]), tile


def far(torch, a, ld):
    """a on the device, column-major with leading dimension ld, NaN between its columns' ends and starts."""
    rows, cols = a.shape
    buf = torch.empty(ld * (cols - 1) + rows, dtype=torch.float64 if a.dtype == np.float64 else torch.float32, device="cuda")
    v = torch.as_strided(buf, (rows, cols), (1, ld))
    for c in range(cols):
        buf[c * ld:c * ld + rows + 64] = float("nan")
    v.copy_(torch.from_numpy(np.ascontiguousarray(a)))
    return v


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("wide", ["A", "B"])
@pytest.mark.parametrize("method", ["f64", "f32", "f32_bf16x3"])
def test_wide_leading_dimensions(gpu, method, wide, ta, tb, tmp_path):
    """Single-problem and grouped products, ragged, in one and in two chunks of k."""
    dt = np.float64 if method == "f64" else np.float32
    m, n, k = 37, 35, 41
    ld = (1 << 32) // (32 * dt().itemsize) + 6  # past the limits of both (grouped: 128 rows of ld elements)
    if (wide == "A" and ta == "T") or (wide == "B" and tb == "N"):
        ld = (1 << 32) // (128 * dt().itemsize) + 6
    A, B, C0 = G.matrix(1, m, k, dtype=dt), G.matrix(2, k, n, dtype=dt), G.matrix(3, m, n, dtype=dt)
    a, b = (x if t == "N" else np.asfortranarray(x.T) for x, t in ((A, ta), (B, tb)))
    a = far(gpu, a, ld) if wide == "A" else to_dev(gpu, a)
    b = far(gpu, b, ld) if wide == "B" else to_dev(gpu, b)
    tol = 2 * k * 2.0**-24 * (np.abs(A).astype(np.float64) @ np.abs(B))
    exact = A.astype(np.float64) @ B
    if method != "f32_bf16x3":
        C = jb.device_matrix(m, n, a.dtype)
        jb.gemm_(ta, tb, 1.0, a, b, 0.0, C)
        assert np.array_equal(bits(to_host(C)), bits(O.jmul(A, B)))
    jb.tune_reset()
    try:
        for splitk in (1, 2):
            write_table(str(tmp_path / f"t{splitk}.json"), method, [(m, n, k)], 0, splitk)
            C = to_dev(gpu, C0)
            jb.gemm_grouped_(method, [GemmDesc(ta, tb, 1.0, a, b, 0.0, C)])
            got = to_host(C)
            if method == "f32_bf16x3":
                assert np.all(np.abs(got - exact) <= tol), splitk
            else:
                ref = O.jmul(A, B) if splitk == 1 else O.jmul(A[:, :32], B[:32]) + O.jmul(A[:, 32:], B[32:])
                assert np.array_equal(bits(got), bits(ref)), splitk
    finally:
        jb.tune_reset()
