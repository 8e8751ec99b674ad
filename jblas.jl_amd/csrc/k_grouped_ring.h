// k_grouped_ring.h -- persistent grouped kernels of the native methods, one per
// tile and transpose combination, and one per combination for leading dimensions
// past 32-bit offsets (instantiated in k_grouped_ring*.hip).
#pragma once
#include "jb_grouped.h"
#include "jb_ring.h"

namespace jb {
namespace {

// Columns coff.. of a BM x ibn item on one ring tile: loads, MFMAs and the result,
// to C through the alpha/beta epilogue or, with several splits, to this split's slab.  FP64 and FP32 chains start from -0.0 and each k-split is one
// fma chain in increasing k, so every split is the jmul! recurrence bit for bit.
template <typename Tile, typename T, bool TA, bool TB, int BM>
__device__ __forceinline__ void ring_part(const GProb& P, const GItem& w, int64_t ms, int64_t n0, int coff, int ibn,
                                          char* ring) {
  constexpr int WIM = Tile::WIM, WIN = Tile::WIN;
  const int64_t ns = n0 + coff, kb = (int64_t)w.split * P.kchunk;
  gptr<const T> A = as_global(static_cast<const T*>(P.A)) + (TA ? kb + ms * P.lda : ms + kb * P.lda);
  gptr<const T> B = as_global(static_cast<const T*>(P.B)) + (TB ? ns + kb * P.ldb : kb + ns * P.ldb);
  Tile tile(ring, threadIdx.x);
  tile.begin(A, P.lda, B, P.ldb, P.m - ms, P.n - ns, min(P.k - kb, P.kchunk));
  typename Tile::Acc acc;
#pragma unroll
  for (int i = 0; i < WIM; ++i)
#pragma unroll
    for (int j = 0; j < WIN; ++j) acc[i][j] = typename Tile::acc_t{T(-0.0), T(-0.0), T(-0.0), T(-0.0)};
  // padding is skipped down to 32 x 32 blocks of the tile
  tile.template run_fringe<1, 1>(acc, P.m - ms, P.n - ns);
  if (P.splitk == 1) {
    T* C = static_cast<T*>(P.C) + ms + ns * P.ldc;
    if (P.k == 0) {  // no products (k == 0 or alpha == 0): C = beta*C, +0 for beta == 0
      gptr<T> c = as_global(C);
      const T beta = (T)P.beta;
#pragma unroll 1
      for (int i = 0; i < WIM; ++i)
#pragma unroll 1
        for (int j = 0; j < WIN; ++j)
#pragma unroll 1
          for (int r = 0; r < 4; ++r)
            if (tile.row(i) < P.m - ms && tile.col(j, r) < P.n - ns) {
              gptr<T> e = c + tile.row(i) + tile.col(j, r) * P.ldc;
              *e = beta != T(0) ? beta * *e : T(0);
            }
    } else {
      tile.store(acc, C, P.ldc, P.m - ms, P.n - ns, (T)P.alpha, (T)P.beta);
    }
  } else {
    gptr<T> slab = as_global(static_cast<T*>(P.part)) + ((int64_t)w.tile * P.splitk + w.split) * (BM * ibn);
#pragma unroll
    for (int i = 0; i < WIM; ++i)
#pragma unroll
      for (int j = 0; j < WIN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) agent_store<T>(slab + tile.row(i) + (coff + tile.col(j, r)) * BM, acc[i][j][r]);
  }
}

// Pulls native items of one tile and transpose combination from their
// queues.  Bound: the matrix cores for k from about 256, C's bytes below (1024^2
// problems, 128x64 tile: 70.5 TF/s of 78.6 at k = 1024, 63.5 at 256, 40.7 at 64).
//   RING_TALL   128x64, three workgroups per CU; a 128x128 item runs as two halves
//   RING_WIDE   64x128
//   RING_SMALL  FP32 32x32 (FP32 RING_TALL is 64x64)
// Fringe items multiply only the blocks that reach into C, so FP64 64x64 and 32x32
// tiles run in 128x64 items.  1024-problem log-uniform FP64 set, us: register-staged
// tiles 2890; ring tiles 2640; without the fringes' padding 2500; with the buffer
// stores and cheap tails of jb_ring.h 2465; without kernels for 64x64 and 32x32
// beside these (they took their LDS at a fifth of their rate) 2350.  One kernel for
// all shapes spilled (3005).
template <typename Tile, typename T, bool TA, bool TB, int BM, int BN, int MINW>
__global__ __launch_bounds__(Tile::NTH, MINW) void grouped_ring_kernel(const GProb* __restrict__ probs,
                                                                      const GItem* __restrict__ items,
                                                                      const int* __restrict__ qdesc, int* __restrict__ qnext,
                                                                      int* __restrict__ counters) {
  __shared__ __attribute__((aligned(1024))) char ring[Tile::SMEM];
  __shared__ int s_item, s_flag;
  int q = blockIdx.x % NXCD, tries = 0;
  for (;;) {
    const int it = pop_item(qdesc, qnext, q, tries, &s_item);  // its barriers: every wave is done with the ring
    if (it < 0) break;
    const GItem w = items[it];
    const GProb P = probs[w.prob];
    const int tm = w.tile / P.tiles_n, tn = w.tile % P.tiles_n;
    const int ibn = BM == 128 && P.cfg == CFG_LARGE ? 128 : BN;  // columns of the item
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * ibn;
    for (int c = 0; c < ibn && n0 + c < P.n; c += BN) {
      if (c) __syncthreads();  // every wave is done with the first half's stages
      ring_part<Tile, T, TA, TB, BM>(P, w, m0, n0, c, ibn, ring);
    }
    splitk_combine<T, BM, Tile::NTH>(P, tm, tn, ibn, counters, &s_flag);
  }
}

enum { RING_TALL = 0, RING_WIDE = 1, RING_SMALL = 2 };
template <typename T, bool TA, bool TB>
GroupedKernelFn ring_kernel_of(int which) {
  if constexpr (sizeof(T) == 8) {
    if (which == RING_TALL) return grouped_ring_kernel<RingTile<T, TA, TB, false, 128, 64, 2, 2, 16, 2>, T, TA, TB, 128, 64, 3>;
    return grouped_ring_kernel<RingTile<T, TA, TB, false, 64, 128, 2, 2, 16, 2>, T, TA, TB, 64, 128, 3>;
  } else {
    if (which != RING_SMALL) return grouped_ring_kernel<RingTile<T, TA, TB, false, 64, 64, 2, 2, 32, 2>, T, TA, TB, 64, 64, 4>;
    return grouped_ring_kernel<RingTile<T, TA, TB, false, 32, 32, 2, 2, 32, 3>, T, TA, TB, 32, 32, 4>;
  }
}
template <typename T>
GroupedKernelFn ring_kernel_of(int which, int combo) {
  switch (combo) {
    case 0: return ring_kernel_of<T, false, false>(which);
    case 1: return ring_kernel_of<T, false, true>(which);
    case 2: return ring_kernel_of<T, true, false>(which);
    default: return ring_kernel_of<T, true, true>(which);
  }
}
// 64x64 items with 64-bit offsets
template <typename T>
GroupedKernelFn ring_wide_ld_kernel(int combo) {
  constexpr int BK = sizeof(T) == 8 ? 16 : 32;
  switch (combo) {
    case 0: return grouped_ring_kernel<RingTile<T, false, false, true, 64, 64, 2, 2, BK, 2>, T, false, false, 64, 64, 2>;
    case 1: return grouped_ring_kernel<RingTile<T, false, true, true, 64, 64, 2, 2, BK, 2>, T, false, true, 64, 64, 2>;
    case 2: return grouped_ring_kernel<RingTile<T, true, false, true, 64, 64, 2, 2, BK, 2>, T, true, false, 64, 64, 2>;
    default: return grouped_ring_kernel<RingTile<T, true, true, true, 64, 64, 2, 2, BK, 2>, T, true, true, 64, 64, 2>;
  }
}

}  // namespace
}  // namespace jb
