// jb_grouped.h -- work descriptors and device helpers of the grouped launches
// (jb_grouped.hip, k_grouped_ring*.hip).
#pragma once
#include "jb_internal.h"

namespace jb {

constexpr int GNT = 256;  // 4 waves
// (Operand and result pointers come from problem descriptors in memory: every
// access goes through as_global, jb_internal.h.)
// Work-item configurations: 0 = 64x64 MFMA tile, 1 = 32x32 MFMA tile, 2 = the
// whole problem on the vector ALUs (m, n, k <= SMALL_MAX, one split); FP64 and
// 3xBF16 only: 3 = 128x128, 4 = 128x64, 5 = 64x128 MFMA tiles.
constexpr int NCFG = 6;
constexpr int CFG_BM[NCFG] = {64, 32, 64, 128, 128, 64};  // tile rows
constexpr int CFG_BN[NCFG] = {64, 32, 64, 128, 64, 128};  // tile columns
constexpr int CFG_SMALL = 2;
constexpr int CFG_LARGE = 3;
constexpr int CFG_TALL = 4;
constexpr int CFG_WIDE = 5;
constexpr int SMALL_MAX = 64;
__host__ __device__ constexpr bool large_cfg(int cfg) { return cfg >= CFG_LARGE; }

// Device descriptor of one problem.
struct GProb {
  const void* A;
  const void* B;
  void* C;
  void* part;         // split-K partials: tiles * splitk slabs of BM*BN elements
  int64_t m, n, k, lda, ldb, ldc;
  double alpha, beta;
  int ta, tb, cfg, splitk;
  int tiles_m, tiles_n;
  int64_t kchunk;     // k per split (multiple of 32)
  int counter_base;   // index of this problem's first per-tile arrival counter
  int pad_;
};
struct GItem {
  int prob, tile, split, pad_;
};

typedef void (*GroupedKernelFn)(const GProb*, const GItem*, const int*, int*, int*);
struct GroupedKernel {
  GroupedKernelFn fn;
  int threads;
};
// The persistent kernels of the native methods' MFMA tiles (k_grouped_ring.h) for
// transpose combination 2 ta + tb: `which` tile, or, for leading dimensions past
// 32-bit offsets, 64x64 tiles.
GroupedKernelFn grouped_ring_f64(int which, int combo);
GroupedKernelFn grouped_ring_f64_wide_ld(int combo);
GroupedKernelFn grouped_ring_f32(int which, int combo);
GroupedKernelFn grouped_ring_f32_wide_ld(int combo);
// Those of the 3xBF16 method (k_grouped_x3.hip): 128x128, 128x64, 64x128, 64x64 items.
GroupedKernel grouped_x3(int which, int combo);
GroupedKernelFn grouped_x3_wide_ld(int combo);

namespace {

// The thread index as an opaque value, read once per work item: offsets derived
// from it are then formed inside the work loop of the persistent kernel rather
// than hoisted out of it and held in registers across the items.
__device__ __forceinline__ int work_item_tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// Result element (i, j) of tile (tm, tn): with one split it goes straight to
// C through the alpha/beta epilogue, otherwise to this split's partial slab.
template <typename T, int BM, int BN>
__device__ __forceinline__ void put_result(const GProb& P, int tm, int tn, int split, int i, int j, T v) {
  if (P.splitk == 1) {
    const int64_t m = (int64_t)tm * BM + i, n = (int64_t)tn * BN + j;
    if (m < P.m && n < P.n) {
      gptr<T> C = as_global(static_cast<T*>(P.C));
      T c;
      if (P.k == 0) {  // no products (k == 0 or alpha == 0): C = beta*C, 0 for beta == 0
        c = (T)P.beta != T(0) ? (T)P.beta * C[m + n * P.ldc] : T(0);
      } else {
        c = (T)P.alpha * v;
        if ((T)P.beta != T(0)) c = fma((T)P.beta, C[m + n * P.ldc], c);
      }
      C[m + n * P.ldc] = c;
    }
  } else {
    const int tile = tm * P.tiles_n + tn;
    gptr<T> slab = as_global(static_cast<T*>(P.part)) + ((int64_t)tile * P.splitk + split) * (BM * BN);
    agent_store(slab + i + j * BM, v);
  }
}

// After every thread stored its partials: the last split of the tile to
// arrive sums all partials in split order and applies the epilogue.
template <typename T, int BM, int NTH>
__device__ void splitk_combine(const GProb& P, int tm, int tn, int BN, int* counters, int* sflag) {
  if (P.splitk == 1) return;
  const int tile = tm * P.tiles_n + tn;
  drain_stores();
  __syncthreads();
  if (threadIdx.x == 0) *sflag = atomicAdd(counters + P.counter_base + tile, 1);
  __syncthreads();
  if (*sflag != P.splitk - 1) return;  // not the last split of this tile
  gptr<const T> slab = as_global(static_cast<const T*>(P.part)) + ((int64_t)tile * P.splitk) * (BM * BN);
  gptr<T> C = as_global(static_cast<T*>(P.C));
  const T alpha = (T)P.alpha, beta = (T)P.beta;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  // loads in flight per thread (64- and 128-row tiles have a multiple of 64 columns, the 32-row one 32)
  constexpr int U = BM == 32 ? 4 : 16;
  static_assert(BM * (BM == 32 ? 32 : 64) % (U * NTH) == 0, "whole groups of loads");
  for (int e = threadIdx.x; e < BM * BN; e += U * NTH) {
    T s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) s[u] = agent_load<T>(slab + e + u * NTH);
    for (int q = 1; q < P.splitk; ++q)
#pragma unroll
      for (int u = 0; u < U; ++u) s[u] += agent_load<T>(slab + (int64_t)q * (BM * BN) + e + u * NTH);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = (e + u * NTH) % BM, j = (e + u * NTH) / BM;
      const int64_t m = m0 + i, n = n0 + j;
      if (m < P.m && n < P.n) {
        T c = alpha * s[u];
        if (beta != T(0)) c = fma(beta, C[m + n * P.ldc], c);
        C[m + n * P.ldc] = c;
      }
    }
  }
}

// Work queues of one persistent launch, one per XCD: queue x holds items
// [qdesc[x], qdesc[x] + qdesc[NXCD + x]) of the launch's item array and is
// drained through counter qnext[x].  Workgroups are dispatched to the XCDs
// round-robin, so workgroup b pops from queue b % NXCD first: the tiles that
// share operand panels were put in one queue and meet in one XCD's L2.  Once
// its queue is drained a workgroup takes items from the others in turn.
// Returns the item index, or -1 after every queue was found drained (each
// workgroup then leaves; an item is taken exactly once, by the atomic on its
// queue's counter).
constexpr int NXCD = 8;
__device__ __forceinline__ int pop_item(const int* __restrict__ qdesc, int* __restrict__ qnext, int& q, int& tries,
                                        int* s_item) {
  for (;;) {
    if (threadIdx.x == 0) *s_item = atomicAdd(qnext + q, 1);
    __syncthreads();
    // uniform across the wave: descriptor loads become scalar loads into SGPRs
    const int it = __builtin_amdgcn_readfirstlane(*s_item);
    __syncthreads();
    if (it < qdesc[NXCD + q]) return qdesc[q] + it;
    if (++tries == NXCD) return -1;
    q = (q + 1) % NXCD;
  }
}

}  // namespace
}  // namespace jb
