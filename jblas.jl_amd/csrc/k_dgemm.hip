// k_dgemm.hip -- FP64 and FP32 GEMM kernels for gfx950.
//
// (1) gemm_mfma: C = alpha*op(A)*op(B) + beta*C on v_mfma_f64_16x16x4f64 or
//     v_mfma_f32_16x16x4f32.  Replaces jmul!'s register-tiled AVX loop
//     (src/gemm.jl:244-348): the CPU register tile (pick_kernel_size,
//     src/kernel_structure.jl:76-99) becomes a wave tile of 16x16 MFMA blocks,
//     and the software prefetch (src/memory_management.jl:181-277) an LDS ring
//     that direct global->LDS loads fill ahead of the MFMAs.  op(A)/op(B)
//     transposition is absorbed by the ring's image.
// (2) dgemm_recurrence: one fma chain per element in increasing k, the exact
//     order of src/gemm.jl:86 (first product) and :165 (fma k-step), on the
//     vector ALUs: an independent restatement of (1)'s bits.
#include "jb_ring.h"
#include <algorithm>
#include <cstdlib>
#include <cstring>

namespace jb {
namespace {

// ---------------------------------------------------------------------------
// (1) MFMA GEMM: one block per tile of C (jb_ring.h) and, for the adjoints of a
//     small product, per chunk of k.
// ---------------------------------------------------------------------------

// The kernel's arguments, in one struct: the runtime looks up each pointer that is an argument
// of its own, and a kernel that reads a grid dimension (here splits) takes the implicit arguments
// besides, 256 bytes that the host fills in for every launch.  256^3 FP64 from Python, all of it
// host time, eight processes each: 10.18 us with 17 arguments and the implicit ones, 9.90 so.
template <typename T>
struct KernelArgs {
  int64_t M, N, K;
  T alpha;
  const T* A;
  int64_t lda;
  const T* B;
  int64_t ldb;
  T beta;
  T* C;
  int64_t ldc;
  int tiles_m, tiles_n, acc_from_c;
  int splits;       // gridDim.y
  int64_t kchunk;   // k per split
  T* part;          // the splits' results (null: one split)
  int* counters;    // per tile
};

// Split-K: each block stores its chunk's results, thread by thread, to its slab; the
// last block of the tile to arrive sums the slabs in split order into acc and
// returns true.  The counters are zero between launches: the last block clears its own.
template <typename T, typename Tile>
__device__ __forceinline__ bool splitk_sum(typename Tile::Acc& acc, const KernelArgs<T>& p, int id, char* lds) {
  constexpr int EL = Tile::WIM * Tile::WIN * 4;
  gptr<T> slab = as_global(p.part) + (int64_t)id * p.splits * (EL * Tile::NTH) + threadIdx.x;
  auto at = [&](int q, int i, int j, int r) { return ((int64_t)q * EL + (i * Tile::WIN + j) * 4 + r) * Tile::NTH; };
#pragma unroll
  for (int i = 0; i < Tile::WIM; ++i)
#pragma unroll
    for (int j = 0; j < Tile::WIN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) agent_store(slab + at(blockIdx.y, i, j, r), acc[i][j][r]);
  int* flag = reinterpret_cast<int*>(lds);
  drain_stores();
  __syncthreads();  // (every wave is done with the ring)
  if (threadIdx.x == 0) *flag = atomicAdd(p.counters + id, 1);
  __syncthreads();
  if (*flag != p.splits - 1) return false;
  if (threadIdx.x == 0) p.counters[id] = 0;
#pragma unroll
  for (int i = 0; i < Tile::WIM; ++i)
#pragma unroll
    for (int j = 0; j < Tile::WIN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = agent_load<T>(slab + at(0, i, j, r));
  for (int q = 1; q < p.splits; ++q)
#pragma unroll
    for (int i = 0; i < Tile::WIM; ++i)
#pragma unroll
      for (int j = 0; j < Tile::WIN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] += agent_load<T>(slab + at(q, i, j, r));
  return true;
}

template <typename T, bool TA, bool TB, bool WIDE, int BTM, int BTN, int WGM, int WGN, int BK, int NSLOT,
          int MINW>
__global__ __launch_bounds__(64 * WGM * WGN, MINW) void gemm_mfma_kernel(KernelArgs<T> p) {
  const int64_t M = p.M, N = p.N, K = p.K, lda = p.lda, ldb = p.ldb, ldc = p.ldc;
  T* const C = p.C;
  typedef RingTile<T, TA, TB, WIDE, BTM, BTN, WGM, WGN, BK, NSLOT> Tile;
  constexpr int WIM = Tile::WIM, WIN = Tile::WIN;
  __shared__ __attribute__((aligned(1024))) char ring[Tile::SMEM];

  const int nblocks = p.tiles_m * p.tiles_n;
  const int id = xcd_remap(blockIdx.x, nblocks, 8);
  int tm, tn;
  tile_coords(id, p.tiles_m, p.tiles_n, 8, tm, tn);
  const int64_t m0 = (int64_t)tm * BTM, n0 = (int64_t)tn * BTN, kb = blockIdx.y * p.kchunk;
  Tile tile(ring, threadIdx.x);

  // Chains start from -0.0: the first MFMA step fma(a, x, -0.0) is then exactly
  // fl(a * x) for every input, the plain first product of the reference
  // recurrence (src/gemm.jl:86), signed zeros included (a start of +0.0 would
  // turn an all -0 chain into +0).  Callers route k == 0 elsewhere.
  // acc_from_c (kernel! semantics, src/kernels.jl:225-233): each chain starts
  // from the element of C instead, every k-step an fma; the caller passes
  // alpha = 1, beta = 0, so the epilogue stores the chain value itself.
  constexpr T acc0 = T(-0.0);
  typename Tile::Acc acc;
#pragma unroll
  for (int i = 0; i < WIM; ++i)
#pragma unroll
    for (int j = 0; j < WIN; ++j) acc[i][j] = typename Tile::acc_t{acc0, acc0, acc0, acc0};
  if (p.acc_from_c) {
#pragma unroll
    for (int i = 0; i < WIM; ++i) {
      const int64_t m = m0 + tile.row(i);
#pragma unroll
      for (int j = 0; j < WIN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t n = n0 + tile.col(j, r);
          if (m < M && n < N) acc[i][j][r] = C[m + n * ldc];
        }
    }
  }
  tile.begin(as_global(p.A) + (TA ? kb + m0 * lda : m0 + kb * lda), lda, as_global(p.B) + (TB ? n0 + kb * ldb : kb + n0 * ldb),
             ldb, M - m0, N - n0, upper_half(K - kb - p.kchunk) < 0 ? K - kb : p.kchunk);
  tile.run(acc);
  if (p.part && !splitk_sum<T, Tile>(acc, p, id, ring)) return;
  tile.store(acc, C + m0 + n0 * ldc, ldc, M - m0, N - n0, p.alpha, p.beta);
}

// ---------------------------------------------------------------------------
// (2) Sequential-fma FP64 GEMM (the recurrence on the vector ALUs): 64x64 block
//     tile, each thread a 4x4 register tile, BK=16 LDS stage.
// ---------------------------------------------------------------------------
constexpr int NT = 256;      // threads per block
constexpr int BK = 16;       // k extent of one LDS stage
constexpr int RB = 64;       // tile rows and columns
constexpr int RSTRIDE = 66;  // LDS row stride in doubles

// One RB x BK operand tile, element by element: registers, then LDS k-major.
//   RC: element (r, kk) at P[(r0+r) + (k0+kk)*ld] (A 'N', B 'T'), else at P[(k0+kk) + (r0+r)*ld]
template <bool RC>
struct TileLoader {
  static constexpr int PER = RB * BK / NT;
  double v[PER];
  static __device__ __forceinline__ int row(int e) { return RC ? e % RB : e / BK; }
  static __device__ __forceinline__ int kof(int e) { return RC ? e / RB : e % BK; }
  __device__ __forceinline__ void load(const double* __restrict__ P, int64_t ld, int64_t r0, int64_t k0, int64_t Rtot,
                                       int64_t K) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = threadIdx.x + NT * i;
      const int64_t r = r0 + row(e), k = k0 + kof(e);
      v[i] = (r < Rtot && k < K) ? P[RC ? r + k * ld : k + r * ld] : 0.0;
    }
  }
  __device__ __forceinline__ void store(double* S) const {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = threadIdx.x + NT * i;
      S[kof(e) * RSTRIDE + row(e)] = v[i];
    }
  }
};

template <bool TA, bool TB>
__global__ __launch_bounds__(NT, 2) void dgemm_recurrence_kernel(int64_t M, int64_t N, int64_t K, double alpha,
                                                                 const double* __restrict__ A, int64_t lda,
                                                                 const double* __restrict__ B, int64_t ldb, double beta,
                                                                 double* __restrict__ C, int64_t ldc, int tiles_m,
                                                                 int tiles_n) {
  typedef double T;
  __shared__ __attribute__((aligned(16))) T As[BK * RSTRIDE];
  __shared__ __attribute__((aligned(16))) T Bs[BK * RSTRIDE];
  const int nblocks = tiles_m * tiles_n;
  const int tile = xcd_remap(blockIdx.x, nblocks, 8);
  int tm, tn;
  tile_coords(tile, tiles_m, tiles_n, 8, tm, tn);
  const int64_t m0 = (int64_t)tm * RB, n0 = (int64_t)tn * RB;
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;

  TileLoader<!TA> la;
  TileLoader<TB> lb;
  T acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[i][j] = T(0);
    }

  for (int64_t k0 = 0; k0 < K; k0 += BK) {
    la.load(A, lda, m0, k0, M, K);
    lb.load(B, ldb, n0, k0, N, K);
    __syncthreads();  // previous stage fully consumed
    la.store(As);
    lb.store(Bs);
    __syncthreads();
    const int kmax = (int)min<int64_t>(BK, K - k0);
    int kk = 0;
    if (k0 == 0) {  // acc_1 = fl(a_1 * x_1)   (src/gemm.jl:86)
      T a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[tx + 16 * i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[ty + 16 * j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = a[i] * b[j];
      kk = 1;
    }
    for (; kk < kmax; ++kk) {  // acc_n = fma(a_n, x_n, acc_{n-1})   (src/gemm.jl:165)
      T a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk * RSTRIDE + tx + 16 * i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[kk * RSTRIDE + ty + 16 * j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fma(a[i], b[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t m = m0 + tx + 16 * i, n = n0 + ty + 16 * j;
      if (m < M && n < N) {
        T c = alpha * acc[i][j];
        if (beta != T(0)) c = fma(beta, C[m + n * ldc], c);
        C[m + n * ldc] = c;
      }
    }
}

template <typename T>
__global__ void scale_kernel(int64_t m, int64_t n, T beta, T* __restrict__ C, int64_t ldc) {
  const int64_t total = m * n;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = idx % m, j = idx / m;
    T* p = C + i + j * ldc;
    *p = (beta == T(0)) ? T(0) : beta * *p;
  }
}


}  // namespace

int gemm_splits(const GemmArgs& g) { return g.kchunk > 0 ? (int)std::max<int64_t>(1, (g.k + g.kchunk - 1) / g.kchunk) : 1; }

template <typename T, bool WIDE, int BTM, int BTN, int WGM, int WGN, int BK, int NSLOT, int MINW>
static hipError_t launch_gemm_mfma_bt(const GemmArgs& g, hipStream_t s, int acc_from_c) {
  const int tiles_m = (int)((g.m + BTM - 1) / BTM), tiles_n = (int)((g.n + BTN - 1) / BTN);
  const int nblocks = tiles_m * tiles_n;
  const int splits = gemm_splits(g);
  const KernelArgs<T> args = {g.m, g.n, g.k, (T)g.alpha, static_cast<const T*>(g.A), g.lda, static_cast<const T*>(g.B), g.ldb,
                              (T)g.beta, static_cast<T*>(g.C), g.ldc, tiles_m, tiles_n, acc_from_c, splits,
                              splits > 1 ? g.kchunk : g.k, static_cast<T*>(g.part), g.counters};
  const char* tname = sizeof(T) == 8 ? "dgemm_mfma" : "sgemm_mfma";
#define JB_LAUNCH(TA, TB)                                                                                             \
  hipLaunchKernelGGL((gemm_mfma_kernel<T, TA, TB, WIDE, BTM, BTN, WGM, WGN, BK, NSLOT, MINW>), dim3(nblocks, splits), \
                     dim3(64 * WGM * WGN), 0, s, args)
  timing_begin(s, tname);
  if (!g.ta && !g.tb) JB_LAUNCH(false, false);
  else if (!g.ta && g.tb) JB_LAUNCH(false, true);
  else if (g.ta && !g.tb) JB_LAUNCH(true, false);
  else JB_LAUNCH(true, true);
#undef JB_LAUNCH
  timing_end(s, tname);
  return hipGetLastError();
}

// Ring configuration <waves along m, along n, k per stage, slots, waves per SIMD> of each tile.  A stage is 16 KB
// (FP64 64-tile) to 32 KB; 128- and 64-tiles keep two slots and several workgroups per CU, whose waves fill each
// other's barriers, the smaller tiles more slots, since their stages are shorter than a load's latency.  FP64 32x32, us
// with four slots of 16 k, three of 16 and three of 32: 128^3 4.05, 4.09 and 3.99, 256^3 5.08, 5.03 and 5.32, 512^3
// 7.21, 7.31 and 7.48, 768^3 20.2, 21.7 and 20.5.
template <typename T, int BTM, int BTN> struct Ring;
template <> struct Ring<double, 128, 128> { static constexpr auto run = launch_gemm_mfma_bt<double, false, 128, 128, 2, 4, 16, 2, 4>; };
template <> struct Ring<double, 64, 64> { static constexpr auto run = launch_gemm_mfma_bt<double, false, 64, 64, 2, 2, 16, 2, 4>; };
template <> struct Ring<double, 64, 32> { static constexpr auto run = launch_gemm_mfma_bt<double, false, 64, 32, 2, 2, 16, 3, 4>; };
template <> struct Ring<double, 32, 32> { static constexpr auto run = launch_gemm_mfma_bt<double, false, 32, 32, 2, 2, 16, 4, 4>; };
template <> struct Ring<float, 128, 128> { static constexpr auto run = launch_gemm_mfma_bt<float, false, 128, 128, 2, 4, 32, 2, 4>; };
template <> struct Ring<float, 64, 64> { static constexpr auto run = launch_gemm_mfma_bt<float, false, 64, 64, 2, 2, 32, 2, 4>; };
template <> struct Ring<float, 64, 32> { static constexpr auto run = launch_gemm_mfma_bt<float, false, 64, 32, 2, 2, 32, 3, 4>; };
template <> struct Ring<float, 32, 32> { static constexpr auto run = launch_gemm_mfma_bt<float, false, 32, 32, 2, 2, 32, 3, 4>; };

// Tile choice: the tile whose fullest CU finishes first.  That CU runs
// ceil(tiles / CUs) tiles, at the tile's own rate: larger tiles read less LDS per
// MFMA and run faster, smaller ones spread a grid more evenly.  Rates relative to
// the 128-tile, measured on full grids (2048^3 to 8192^3); one 128- or 64-tile
// alone on its CU has no other workgroup to fill its barriers (5 and 10 % slower).
// Measured, us (128 / 64 / 64x32 / 32): FP64 512^3 61 / 18.5 / 11.6 / 7.6, 1024^3
// 119 / 38.5 / 34.6 / 34.8, 1536^3 176 / 134 / 114 / 117, 3072^3 1010 / 795 / 832 /
// 888, 4096^3 1798 / 1909 / 1995 / 2192; FP32 800x840x900 56 / 19.0 / 19.1 / 16.9,
// 3072^3 514 / 405 / 434 / 474, 4096^3 908 / 923 / 1003 / 1127.
enum TileId { T128, T64, T64X32, T32, TWIDE };
template <typename T>
static TileId pick_tile(const GemmArgs& g) {
  constexpr bool F64 = sizeof(T) == 8;
  // A load's offset inside a stage spans up to 128 rows of ld elements (k contiguous) or 32 k of them (rows
  // contiguous).  Past 32 bits (from 2^22 or 2^24 doubles on) the 64x32 tile with 64-bit addresses takes the problem.
  const int64_t lim = ((int64_t)1 << 32) / (int64_t)sizeof(T);
  if (g.lda >= lim / (g.ta ? 128 : 32) || g.ldb >= lim / (g.tb ? 32 : 128)) return TWIDE;
  // testing: pin one variant ("128", "64", "64x32", "32")
  const char* force = getenv("JB_GEMM_TILE");
  if (force && *force) {
    if (!strcmp(force, "128")) return T128;
    if (!strcmp(force, "64")) return T64;
    if (!strcmp(force, "64x32")) return T64X32;
    if (!strcmp(force, "32")) return T32;
  }
  const int64_t cus = std::max(runtime_compute_units(), 1), splits = gemm_splits(g);
  auto cost = [&](int bm, int bn, double rate, double alone) {
    const int64_t blocks = ((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn) * splits;
    const int64_t rounds = (blocks + cus - 1) / cus;
    return (double)(rounds * bm * bn) / (rounds == 1 ? rate * alone : rate);
  };
  const double c128 = cost(128, 128, 1.0, 0.95), c64 = cost(64, 64, F64 ? 0.96 : 0.91, 0.90);
  const double c64x32 = cost(64, 32, F64 ? 0.885 : 0.83, 1.0), c32 = cost(32, 32, F64 ? 0.81 : 0.74, 1.0);
  if (c128 <= std::min(c64, std::min(c64x32, c32))) return T128;
  if (c64 <= std::min(c64x32, c32)) return T64;
  return c64x32 < c32 ? T64X32 : T32;
}

template <typename T>
static hipError_t launch_gemm_mfma(const GemmArgs& g, hipStream_t s, int acc_from_c = 0) {
  switch (pick_tile<T>(g)) {
    case T128: return Ring<T, 128, 128>::run(g, s, acc_from_c);
    case T64: return Ring<T, 64, 64>::run(g, s, acc_from_c);
    case T64X32: return Ring<T, 64, 32>::run(g, s, acc_from_c);
    case T32: return Ring<T, 32, 32>::run(g, s, acc_from_c);
    default: return launch_gemm_mfma_bt<T, true, 64, 32, 2, 2, sizeof(T) == 8 ? 16 : 32, 3, 2>(g, s, acc_from_c);
  }
}

void gemm_mfma_split_need(const GemmArgs& g, size_t elt, size_t* part_bytes, int64_t* counters) {
  static const int BM[] = {128, 64, 64, 32, 64}, BN[] = {128, 64, 32, 32, 32};
  const TileId t = elt == 8 ? pick_tile<double>(g) : pick_tile<float>(g);
  *counters = ((g.m + BM[t] - 1) / BM[t]) * ((g.n + BN[t] - 1) / BN[t]);
  *part_bytes = (size_t)*counters * gemm_splits(g) * BM[t] * BN[t] * elt;
}

hipError_t launch_dgemm_mfma(const GemmArgs& g, hipStream_t s) { return launch_gemm_mfma<double>(g, s); }
// kernel!: C = C + A*X with every chain starting from C (g.alpha, g.beta ignored)
hipError_t launch_dgemm_mfma_acc(const GemmArgs& g, hipStream_t s) {
  GemmArgs h = g;
  h.alpha = 1.0;
  h.beta = 0.0;
  return launch_gemm_mfma<double>(h, s, 1);
}
hipError_t launch_sgemm_mfma(const GemmArgs& g, hipStream_t s) { return launch_gemm_mfma<float>(g, s); }

hipError_t launch_dgemm_recurrence(const GemmArgs& g, hipStream_t s) {
  const int tiles_m = (int)((g.m + RB - 1) / RB), tiles_n = (int)((g.n + RB - 1) / RB);
  const int nblocks = tiles_m * tiles_n;
  auto A = static_cast<const double*>(g.A);
  auto B = static_cast<const double*>(g.B);
  auto C = static_cast<double*>(g.C);
#define JB_LAUNCH(TA, TB)                                                                                         \
  hipLaunchKernelGGL((dgemm_recurrence_kernel<TA, TB>), dim3(nblocks), dim3(NT), 0, s, g.m, g.n, g.k, g.alpha, A, \
                     g.lda, B, g.ldb, g.beta, C, g.ldc, tiles_m, tiles_n)
  timing_begin(s, "dgemm_recurrence");
  if (!g.ta && !g.tb) JB_LAUNCH(false, false);
  else if (!g.ta && g.tb) JB_LAUNCH(false, true);
  else if (g.ta && !g.tb) JB_LAUNCH(true, false);
  else JB_LAUNCH(true, true);
#undef JB_LAUNCH
  timing_end(s, "dgemm_recurrence");
  return hipGetLastError();
}

hipError_t launch_scale_f64(int64_t m, int64_t n, double beta, double* C, int64_t ldc, hipStream_t s) {
  if (m == 0 || n == 0) return hipSuccess;
  const int64_t total = m * n;
  const int blocks = (int)std::min<int64_t>((total + 255) / 256, 4096);
  hipLaunchKernelGGL(scale_kernel<double>, dim3(blocks), dim3(256), 0, s, m, n, beta, C, ldc);
  return hipGetLastError();
}
hipError_t launch_scale_f32(int64_t m, int64_t n, float beta, float* C, int64_t ldc, hipStream_t s) {
  if (m == 0 || n == 0) return hipSuccess;
  const int64_t total = m * n;
  const int blocks = (int)std::min<int64_t>((total + 255) / 256, 4096);
  hipLaunchKernelGGL(scale_kernel<float>, dim3(blocks), dim3(256), 0, s, m, n, beta, C, ldc);
  return hipGetLastError();
}

}  // namespace jb
