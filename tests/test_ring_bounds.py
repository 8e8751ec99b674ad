"""The addresses of the MFMA kernels' ring loads, from the kernels' own address functions
compiled for the host: every dword that a load's descriptor lets through lies inside the
operand, and every LDS element that is multiplied holds the right element of it."""
import os
import subprocess

import numpy as np
import pytest

import jblas_amd as jb
from jblas_amd import build as B
from jblas_amd import generators as G
from jblas_amd.grouped import GemmDesc
from oracle import oracle as O

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include <vector>
#include "jb_ring.h"
using namespace jb;

// One operand of `rows` rows from the tile's first on, leading dimension ld, K of k.
template <typename T, int R, int BK, bool RC, int NW>
int check(int64_t rows, int64_t ld, int64_t K) {
  typedef RingOperand<T, R, BK, RC, NW, false> O;
  constexpr int EB = sizeof(T), VW = 16 / EB;
  const int nst = (int)((K + BK - 1) / BK), nfull = (int)(K / BK);
  const int64_t end = O::extent(ld, rows, K) * EB;
  const int rmax = (int)std::min<int64_t>(RC ? (rows - 1) / VW * VW : rows - 1, R);
  const int64_t kmax = RC ? K - 1 : (K - 1) / VW * VW;
  for (int st = 0; st < nst; ++st) {
    const bool tail = st >= nfull;
    const int64_t k0 = (int64_t)st * BK, base = (RC ? k0 * ld : k0) * EB;
    const int kleft = tail ? (int)(kmax - k0) : BK;
    // RingTile::issue: records of the last stage and, where it can reach the end, of the one before
    const uint32_t records = st == nst - 1 || (O::REACH && st == nst - 2) ? (uint32_t)(O::extent(ld, rows, K - k0) * EB) : ~0u;
    std::vector<int64_t> lds(R * BK, -1);  // byte of the operand in each LDS element, -1: zeros
    for (int wave = 0; wave < NW; ++wave)
      for (int lane = 0; lane < 64; ++lane) {
        O o;
        o.init(ld, rmax, wave, lane);
        for (int i = 0; i < O::NP; ++i) {
          const int p = wave + NW * i;
          const int kp = tail ? O::template krow<true>(p, kleft) : O::template krow<false>(p, kleft);
          const int64_t at = o.off[i] - (tail ? O::past(p, kp, kleft, ld, lane) : 0) + (int64_t)kp * ld * EB;
          for (int d = 0; d < 16; d += 4) {
            if (at + d + 4 > records) continue;
            if (at < 0 || base + at + d + 4 > end)
              return printf("%d-byte elements, R %d, RC %d, waves %d: rows %ld ld %ld K %ld stage %d reads byte %ld of %ld\n",
                            EB, R, RC, NW, (long)rows, (long)ld, (long)K, st, (long)(base + at + d), (long)end), 1;
            if (d % EB == 0) lds[(p * O::PB + lane * 16 + d) / EB] = base + at + d;
          }
        }
      }
    for (int r = 0; r < std::min<int64_t>(rows, R); ++r)
      for (int k = 0; k < std::min<int64_t>(BK, K - k0); ++k)
        if (lds[O::at(r, k)] != (RC ? r + (k0 + k) * ld : k0 + k + r * ld) * EB)
          return printf("%d-byte elements, R %d, RC %d, waves %d: rows %ld ld %ld K %ld stage %d element %d, %d\n", EB, R, RC,
                        NW, (long)rows, (long)ld, (long)K, st, r, k), 1;
  }
  return 0;
}

template <typename T, int R, int NW>
int tile() {
  constexpr int BK = sizeof(T) == 8 ? 16 : 32;
  for (int64_t rows : {1, 2, 3, 4, 5, R - 1, R, R + 1, 2 * R})
    for (int64_t pad : {0, 1, 2, 5})
      for (int64_t K : {1, 2, 3, BK - 1, BK, BK + 1, BK + 2, BK + 3, 2 * BK, 2 * BK + 1, 2 * BK + 2, 3 * BK + 1, 3 * BK + 7})
        if (check<T, R, BK, true, NW>(rows, rows + pad, K) || check<T, R, BK, false, NW>(rows, K + pad, K)) return 1;
  return 0;
}

int main() {
  // the extents and wave counts of the single-problem and grouped tiles
  return tile<double, 128, 8>() || tile<double, 128, 4>() || tile<double, 64, 4>() || tile<double, 32, 4>() ||
         tile<float, 128, 8>() || tile<float, 64, 4>() || tile<float, 32, 4>();
}
"""


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
def test_ring_loads_stay_inside_the_operand(tmp_path):
    src, exe = tmp_path / "ring.hip", tmp_path / "ring"
    src.write_text(PROGRAM)
    subprocess.run([B.HIPCC, "--cuda-host-only", "-std=c++17", "-O1", "-w", "-I", B.CSRC, str(src), "-o", str(exe)], check=True,
                   timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout


def exact_buffer(torch, a, pad):
    """a on the device, leading dimension rows + pad, in a buffer that ends with its last element."""
    rows, cols = a.shape
    ld = rows + pad
    buf = torch.full((ld * (cols - 1) + rows,), float("nan"), dtype=getattr(torch, str(a.dtype)), device="cuda")
    v = torch.as_strided(buf, (rows, cols), (1, ld))
    v.copy_(torch.from_numpy(np.ascontiguousarray(a)))
    return v


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("pad", [0, 1])
def test_one_row_operands(gpu, dtype, pad):
    """Leading dimensions below a vector's length (op(A) of one row, op(B) of one column), k just past whole stages:
    bit for bit the oracle's recurrence, single and grouped."""
    for m, n in ((1, 1), (1, 70), (70, 1), (2, 2)):
        for k in (17, 33, 34, 65, 66, 67):
            A, X = G.matrix(m + k, m, k, dtype=dtype), G.matrix(n + k, k, n, dtype=dtype)
            ref = O.jmul(A, X)
            a, x = exact_buffer(gpu, A, pad), exact_buffer(gpu, np.asfortranarray(X.T), pad)
            D, E = (jb.device_matrix(m, n, a.dtype) for _ in range(2))
            jb.gemm_("N", "T", 1.0, a, x, 0.0, D)
            jb.gemm_grouped_("f64" if dtype == np.float64 else "f32", [GemmDesc("N", "T", 1.0, a, x, 0.0, E)])
            for got in (D, E):
                assert np.array_equal(got.cpu().numpy(), ref), (m, n, k)
