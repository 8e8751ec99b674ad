"""The grouped 3xBF16 tiles at their edges: extents around the tiles and the 32-k
stages, stages masked at the end of k, vectors that start off a 16-byte boundary or end
past the operand, NaN around every operand, splits, leading dimensions past 32-bit
offsets.  |C - C*| <= 2 K 2^-24 (|alpha| |A| |B| + |beta| |C0|) against the FP64 product."""
import numpy as np
import pytest

import jblas_amd as jb
from jblas_amd import generators as G
from jblas_amd.grouped import GemmDesc

from conftest import to_host
from test_grouped_gpu import write_table

pytestmark = pytest.mark.gpu

SHAPES = [(65, 1, 1), (1, 66, 31), (63, 65, 32), (64, 64, 66), (66, 97, 63), (127, 129, 95), (130, 31, 130), (129, 200, 33)]


def placed(torch, a, pad, shift):
    """a column-major with leading dimension rows + pad, `shift` elements off an aligned base, NaN around it."""
    rows, cols = a.shape
    buf = torch.full((shift + (rows + pad) * (cols - 1) + rows,), float("nan"), dtype=torch.float32, device="cuda")
    v = torch.as_strided(buf, (rows, cols), (1, rows + pad), shift)
    v.copy_(torch.from_numpy(np.ascontiguousarray(a)))
    return v


def check(ta, tb, A, B, C0, got, alpha=1.5, beta=0.5):
    a, b = (x.T if t == "T" else x for x, t in ((A.astype(np.float64), ta), (B.astype(np.float64), tb)))
    tol = 2 * a.shape[1] * 2.0**-24 * (abs(alpha) * np.abs(a) @ np.abs(b) + abs(beta) * np.abs(C0))
    assert np.all(np.abs(got - (alpha * a @ b + beta * C0)) <= tol), (ta, tb, a.shape, b.shape)


@pytest.mark.parametrize("cfg", [0, 1, 3, 4, 5])
@pytest.mark.parametrize("splitk", [1, 2])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_x3_tiles_edges(gpu, cfg, splitk, beta, tmp_path):
    jb.tune_reset()
    write_table(str(tmp_path / "t.json"), "f32_bf16x3", SHAPES, cfg, splitk)
    try:
        for ta in "NT":
            for tb in "NT":
                host, descs = [], []
                for i, (m, n, k) in enumerate(SHAPES):
                    A = G.matrix(10 + i, *((m, k) if ta == "N" else (k, m)), dtype=np.float32)
                    B = G.matrix(30 + i, *((k, n) if tb == "N" else (n, k)), dtype=np.float32)
                    C = G.matrix(50 + i, m, n, dtype=np.float32)
                    host.append((A, B, C))
                    descs.append(GemmDesc(ta, tb, 1.5, placed(gpu, A, i % 4, i % 3), placed(gpu, B, i % 2, i % 4), beta,
                                          placed(gpu, C, 1, 0)))
                jb.gemm_grouped_("f32_bf16x3", descs)
                for (A, B, C), d in zip(host, descs):
                    check(ta, tb, A, B, C, to_host(d.C), beta=beta)
                    buf = d.C._base
                    assert int(buf.isnan().sum()) == buf.numel() - C.size  # nothing stored around C
    finally:
        jb.tune_reset()


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "T")])
def test_x3_wide_leading_dimension(gpu, ta, tb):
    m, n, k, ld = 70, 3, 3, (1 << 23) + 1
    sa, sb = ((m, k) if ta == "N" else (k, m)), ((k, n) if tb == "N" else (n, k))
    A, B, C = G.matrix(1, *sa, dtype=np.float32), G.matrix(2, *sb, dtype=np.float32), G.matrix(3, m, n, dtype=np.float32)
    dA, dB, dC = placed(gpu, A, ld - sa[0], 0), placed(gpu, B, 0, 0), placed(gpu, C, 0, 0)
    jb.gemm_grouped_("f32_bf16x3", [GemmDesc(ta, tb, 1.5, dA, dB, 0.5, dC)])
    check(ta, tb, A, B, C, to_host(dC))


def test_large_group_takes_tiles_by_padding(gpu):
    """Past 32 64x128 tiles per compute unit each problem takes the tile with the least padding."""
    m, n, k = 128, 512, 32
    d = GemmDesc("N", "N", 1.0, jb.device_matrix(m, k, gpu.float32), jb.device_matrix(k, n, gpu.float32), 0.0,
                 jb.device_matrix(m, n, gpu.float32))
    cus = jb.device_info()["compute_units"]
    many = -(-32 * cus // 8)
    assert {c[0] for c in jb.grouped_choices("f32_bf16x3", [d] * many)} == {"128x128"}
    assert {c[0] for c in jb.grouped_choices("f32_bf16x3", [d] * (many - 1))} == {"64x128"}
