// jb_grouped.hip -- batched / grouped GEMM in one persistent launch, hipGraph
// plans, the autotuner, and the gemm! pullback.
//
// The reference has no batching: its blocking is static (pick_kernel_size,
// src/kernel_structure.jl:76-99; blocking_structure, src/memory_management.jl:
// 78-140, which nothing calls).  Here every problem of a group gets a tile
// shape and a split-K factor from a measured table (autotuner), and all
// problems run in ONE persistent launch:
//   * work items (problem, output tile, k-split) sorted by decreasing cost
//     are pulled from a device counter by a grid of CU-filling workgroups,
//     so uneven problems load-balance;
//   * the MFMA tiles run in persistent kernels per tile shape and transpose
//     combination (k_grouped_ring.h, k_grouped_x3.hip), the small problems in one
//     more; a plan's kernels run concurrently;
//   * split-K partials go to a workspace slot per (tile, split); the last
//     split to finish (per-tile arrival counter) sums them in split order,
//     so results are deterministic;
//   * methods: FP64 on FP64 MFMA, FP32 on FP32 MFMA, FP32 as 3xBF16 (split on
//     the fly into hi/mid/lo BF16 planes in LDS, 6 products on BF16 MFMA).
// A plan uploads descriptors once and captures [counter reset kernel,
// persistent kernels] in a hipGraph; launching the plan replays the graph.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <type_traits>
#include <vector>

#include "jb_grouped.h"
#include "jb_runtime.h"

namespace jb {
namespace {

// Small problem (m, n, k <= 64) in one work item, the form of fastmul!
// (src/kernels.jl:202-208, kernel_quote :42-201): no MFMA tile; lane = row of C
// (rows >= m recompute row m-1 and store nothing), wave w holds columns
// 16w..16w+15 in registers.  The workgroup first stages all of op(B) (k x n)
// in LDS, [p][j] with rows of SB_STRIDE elements, in two batches of loads;
// each lane then reads its row of op(A) in register chunks of 4 k (the next
// chunk in flight) and B(p, j0..j0+15) as LDS broadcasts, 8 columns at a time.
// Each element is the chain
// acc = A(i,0) B(0,j), acc = fma(A(i,p), B(p,j), acc) for p = 1..k-1 -- the
// plain first product of src/gemm.jl:86 and the k-steps of :165 -- then the
// alpha/beta epilogue of the tiles (put_result).
template <typename T, bool TA, bool TB>
__device__ __forceinline__ void small_tile(const GProb& P, char* smem) {
  constexpr int SC = 16;                          // columns per wave
  constexpr int SB_STRIDE = 64 + 16 / sizeof(T);  // 16-byte aligned rows, 4-way at most on the staging writes
  constexpr int AC = 4;                           // k per register chunk of A
  T* Bs = reinterpret_cast<T*>(smem);
  const int tid = work_item_tid();
  const int lane = tid % 64, wave = tid / 64;
  const int64_t m = P.m, n = P.n, k = P.k;
  gptr<const T> A = as_global(static_cast<const T*>(P.A));
  gptr<const T> B = as_global(static_cast<const T*>(P.B));
  // stage op(B): element e = tid + 256 q is (p, j) with the contiguous index fastest
  constexpr int NQ = 64 * 64 / GNT;  // 16 elements per thread, staged 8 at a time
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    T v[NQ / 2];
#pragma unroll
    for (int q = 0; q < NQ / 2; ++q) {
      const int e = tid + GNT * (q + h * NQ / 2);
      const int pp = TB ? e / 64 : e % 64, jj = TB ? e % 64 : e / 64;
      v[q] = (pp < k && jj < n) ? (TB ? B[jj + (int64_t)pp * P.ldb] : B[pp + (int64_t)jj * P.ldb]) : T(0);
    }
#pragma unroll
    for (int q = 0; q < NQ / 2; ++q) {
      const int e = tid + GNT * (q + h * NQ / 2);
      const int pp = TB ? e / 64 : e % 64, jj = TB ? e % 64 : e / 64;
      Bs[pp * SB_STRIDE + jj] = v[q];
    }
  }
  const int64_t i = lane < m ? lane : m - 1;
  gptr<const T> arow = TA ? A + i * P.lda : A + i;  // A(i, p) = arow[p * astep]
  const int64_t astep = TA ? 1 : P.lda;
  T a[2][AC];
#pragma unroll
  for (int u = 0; u < AC; ++u) a[0][u] = u < k ? arow[u * astep] : T(0);
  __syncthreads();
  const int j0 = SC * wave;
  if (j0 >= n || k == 0) {
    if (k == 0 && j0 < n && lane < m) {  // alpha == 0 or k == 0: C = beta*C, 0 for beta == 0
      gptr<T> C = as_global(static_cast<T*>(P.C));
#pragma unroll
      for (int c = 0; c < SC; ++c)
        if (j0 + c < n) {
          gptr<T> cp = C + i + (j0 + c) * P.ldc;
          *cp = (T)P.beta != T(0) ? (T)P.beta * *cp : T(0);
        }
    }
    return;  // no barrier below
  }
  const T* bp = Bs + j0;
  T acc[SC];
#pragma unroll
  for (int c0 = 0; c0 < SC; c0 += 8) {  // p = 0: the plain first product
    T b[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) b[c] = bp[c0 + c];
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c0 + c] = a[0][0] * b[c];
  }
  // chunks of AC k, two per iteration so that the register buffer of a chunk
  // (cb & 1) is a compile-time index; chunk cb+1 is loaded while cb computes
#pragma unroll 1
  for (int ch = 0; ch * AC < k; ch += 2) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // guarded bodies, no break: the loops unroll fully
      const int cb = ch + h;
      if (cb * AC < k) {
        if ((cb + 1) * AC < k) {
#pragma unroll
          for (int u = 0; u < AC; ++u) {
            const int64_t pn = (int64_t)(cb + 1) * AC + u;
            a[h ^ 1][u] = pn < k ? arow[pn * astep] : T(0);
          }
        }
#pragma unroll
        for (int u = 0; u < AC; ++u) {
          const int pp = cb * AC + u;
          if (pp > 0 && pp < k) {
            const T* brow = bp + pp * SB_STRIDE;
#pragma unroll
            for (int c0 = 0; c0 < SC; c0 += 8) {
              T b[8];
#pragma unroll
              for (int c = 0; c < 8; ++c) b[c] = brow[c0 + c];
#pragma unroll
              for (int c = 0; c < 8; ++c) acc[c0 + c] = fma(a[h][u], b[c], acc[c0 + c]);
            }
          }
        }
      }
    }
  }
  if (lane >= m) return;
  gptr<T> C = as_global(static_cast<T*>(P.C));
  const T alpha = (T)P.alpha, beta = (T)P.beta;
#pragma unroll
  for (int c = 0; c < SC; ++c) {
    const int64_t j = j0 + c;
    if (j < n) {
      T v = alpha * acc[c];
      if (beta != T(0)) v = fma(beta, C[i + j * P.ldc], v);
      C[i + j * P.ldc] = v;
    }
  }
}

template <int KIND>
__device__ __forceinline__ void run_small(const GProb& P, int combo, char* smem) {
  typedef typename std::conditional<KIND == 0, double, float>::type T;
  switch (combo) {
    case 0: small_tile<T, false, false>(P, smem); break;
    case 1: small_tile<T, false, true>(P, smem); break;
    case 2: small_tile<T, true, false>(P, smem); break;
    default: small_tile<T, true, true>(P, smem); break;
  }
}

// The small items.  KIND 0: FP64, 1: FP32.
template <int KIND>
__global__ __launch_bounds__(GNT, 2) void grouped_kernel(const GProb* __restrict__ probs, const GItem* __restrict__ items,
                                                         const int* __restrict__ qdesc, int* __restrict__ qnext,
                                                         int* __restrict__) {
  constexpr int E = KIND == 0 ? 8 : 4;
  __shared__ __attribute__((aligned(16))) char smem[64 * (64 + 16 / E) * E];  // op(B)
  __shared__ int s_item;
  int q = blockIdx.x % NXCD, tries = 0;
  for (;;) {
    const int it = pop_item(qdesc, qnext, q, tries, &s_item);  // its barriers: the previous item's op(B) is read
    if (it < 0) break;
    const GProb P = probs[items[it].prob];
    run_small<KIND>(P, (P.ta ? 2 : 0) + (P.tb ? 1 : 0), smem);
  }
}


int kind_of(int method) {
  if (method == JB_F64_NATIVE) return 0;
  if (method == JB_F32_NATIVE) return 1;
  if (method == JB_F32_BF16X3) return 2;
  return -1;
}

// ---------------------------------------------------------------------------
// autotuning table
// ---------------------------------------------------------------------------
struct TuneEntry {
  int cfg, splitk;
  double ms;
};
std::map<std::string, TuneEntry> g_table;

int ilog2(int64_t x) {
  int r = 0;
  while (x > 1) {
    x >>= 1;
    ++r;
  }
  return r;
}
// Size bucket: (log2 of the geometric mean of m and n, log2 k).
std::string bucket_key(int method, int64_t m, int64_t n, int64_t k) {
  const int mn = ilog2((int64_t)std::sqrt((double)std::max<int64_t>(m, 1) * (double)std::max<int64_t>(n, 1)));
  char buf[64];
  snprintf(buf, sizeof buf, "m%d|mn%d|k%d", method, mn, ilog2(std::max<int64_t>(k, 1)));
  return buf;
}

// Static defaults (no table entry).  Tile: the small path for m, n, k <= 64
// (one work item, B staged in LDS: on 1024 such problems it measured 43.0 us
// against 44.4 us for the tiles in FP64 and 34.7 against 37.6 us in 3xBF16);
// otherwise, for FP64, the tile with the least padded area per unit of
// measured throughput (TILE_RATE: each tile's FP64 rate on groups of
// 1024 x 1024 problems with k = 256 and 1024, relative to the 128x128 tile);
// for 3xBF16 the 64x128 tile (plan_choices refines it for large groups);
// for native FP32 the 64x64 tile from max(m, n) >= 96, else 32x32.
// Split-K is not chosen per problem: plan_build splits the longest work items
// when the whole group has fewer work items than the device holds workgroups
// (the blocking decision that depends on the device, blocking_structure's role
// in src/memory_management.jl:78-140).
// (3xBF16: 170, 155, 156 and 143 TF/s on 1024^3 with the 128x128, 128x64, 64x128 and 64x64
// tile, 127, 118, 119 and 109 with k = 256.)
constexpr double TILE_RATE[2][NCFG] = {{0.90, 0.65, 0.0, 1.0, 1.0, 0.97}, {0.87, 0.0, 0.0, 1.0, 0.92, 0.94}};
int tile_by_rate(int kind, int64_t m, int64_t n) {
  int cfg = CFG_LARGE;
  double best = 0;
  for (int c : {CFG_LARGE, CFG_TALL, CFG_WIDE, 0, 1}) {
    if (kind == 2 && c == 1) continue;  // (the 64x64 tile's kernel)
    const double padded = (double)((m + CFG_BM[c] - 1) / CFG_BM[c] * CFG_BM[c]) *
                          (double)((n + CFG_BN[c] - 1) / CFG_BN[c] * CFG_BN[c]);
    const double t = padded / TILE_RATE[kind / 2][c];
    if (c == CFG_LARGE || t < best) {
      best = t;
      cfg = c;
    }
  }
  return cfg;
}
void default_choice(int kind, int64_t m, int64_t n, int64_t k, int& cfg, int& splitk) {
  splitk = 1;
  if (m <= SMALL_MAX && n <= SMALL_MAX && k <= SMALL_MAX) {
    cfg = CFG_SMALL;
    return;
  }
  if (kind == 1) {
    cfg = std::max(m, n) >= 96 ? 0 : 1;
    return;
  }
  if (kind == 2) cfg = CFG_WIDE;
  else cfg = tile_by_rate(kind, m, n);
}

// A choice taken from a bucket (table, tuner trial, forced) may name the small
// path for a problem that does not fit it: such a problem takes the 32x32 tile;
// the 128-row/column tiles exist for FP64 and 3xBF16 (native FP32 takes 64x64).
void fit_choice(int kind, int64_t m, int64_t n, int64_t k, int& cfg, int& splitk) {
  if (cfg == CFG_SMALL) {
    if (m <= SMALL_MAX && n <= SMALL_MAX && k <= SMALL_MAX) splitk = 1;
    else cfg = 1;
  }
  if (large_cfg(cfg) && kind == 1) cfg = 0;
}

// Returns true when the choice is the static default (plan_build may then add split-K).
bool choose(int method, int64_t m, int64_t n, int64_t k, int& cfg, int& splitk) {
  const int kind = kind_of(method);
  auto it = g_table.find(bucket_key(method, m, n, k));
  bool dflt = false;
  if (it != g_table.end()) {
    cfg = it->second.cfg;
    splitk = it->second.splitk;
  } else {
    default_choice(kind, m, n, k, cfg, splitk);
    dflt = true;
  }
  fit_choice(kind, m, n, k, cfg, splitk);
  return dflt;
}

// ---------------------------------------------------------------------------
// plans
// ---------------------------------------------------------------------------
// Persistent launches of a plan, by kernel: for each tile (ring_of; 3xBF16: grouped_x3)
// one per transpose combination, then one per combination for leading dimensions past
// 32-bit offsets, then one for the small items.
constexpr int L_WIDE = 4 * 4, L_OTHER = L_WIDE + 4, NLAUNCH = L_OTHER + 1;

// forced choice for the autotuner's trial launches: cfg >= 0 forces one choice
// on every problem; otherwise `over` (bucket -> choice) is consulted before the table
struct Forced {
  int cfg = -1, splitk = 1;
  const std::map<std::string, TuneEntry>* over = nullptr;
};

}  // namespace

struct GroupedPlanImpl {
  int method = 0, kind = 0;
  int nitems = 0, nprobs = 0, ncounters = 0;
  // items and grid of each launch (see NLAUNCH)
  int litems[NLAUNCH] = {}, lgrid[NLAUNCH] = {};
  void* dev = nullptr;  // probs | items | queue descriptors | counters | partials
  size_t dev_bytes = 0;
  GProb* probs = nullptr;
  GItem* items = nullptr;
  int* qdesc = nullptr;  // per launch: NXCD queue offsets into items, then NXCD queue lengths
  int* next = nullptr;   // per launch NXCD queue counters, then per-tile arrival counters (zeroed every launch)
  // the persistent launches run concurrently: all but the first on side
  // streams forked from the caller's stream after the counter reset and
  // joined back to it (a launch's tail overlaps the others' work)
  int nside = 0;
  hipStream_t side[NLAUNCH - 1] = {};
  hipEvent_t fork = nullptr, join[NLAUNCH - 1] = {};
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  hipStream_t cap = nullptr;
  // recorded after every replay: the next replay (on any stream) waits for it,
  // since all replays share the work and arrival counters
  hipEvent_t done = nullptr;
  bool launched = false;
  double flops = 0;
};

}  // namespace jb

struct jb_grouped_plan {
  jb::GroupedPlanImpl impl;
};

namespace jb {
namespace {

std::vector<jb_grouped_plan*> g_plans;

int validate_descs(int method, int64_t count, const jb_gemm_desc* d) {
  if (kind_of(method) < 0) return fail(-1, "method must be JB_F64_NATIVE, JB_F32_NATIVE or JB_F32_BF16X3");
  if (count < 0) return fail(-2, "count < 0");
  if (count > 0 && !d) return fail(-3, "descs is NULL");
  if (count > (1 << 24)) return fail(-2, "count above 2^24");
  for (int64_t i = 0; i < count; ++i) {
    GemmArgs g;
    const jb_gemm_desc& x = d[i];
    int rc = validate_gemm(x.transA, x.transB, x.m, x.n, x.k, x.alpha == 0.0, x.A, x.lda, x.B, x.ldb, x.C, x.ldc, &g);
    if (rc) return fail(-3, "descs[%lld]: %s", (long long)i, jb_last_error());
  }
  return JB_OK;
}

size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

// The kernel of launch L (see NLAUNCH) of a plan of method kind `kind`.
GroupedKernel launch_kernel(int kind, int L) {
  if (L == L_OTHER) return {kind == 0 ? grouped_kernel<0> : grouped_kernel<1>, GNT};
  if (kind == 2) return L >= L_WIDE ? GroupedKernel{grouped_x3_wide_ld(L - L_WIDE), GNT} : grouped_x3(L / 4, L % 4);
  if (L >= L_WIDE) return {kind == 0 ? grouped_ring_f64_wide_ld(L - L_WIDE) : grouped_ring_f32_wide_ld(L - L_WIDE), GNT};
  return {kind == 1 ? grouped_ring_f32(L / 4, L % 4) : grouped_ring_f64(L / 4, L % 4), GNT};
}

// Byte offsets inside an operand stage (up to 128 rows or 32 k of ld elements) past 32 bits.
bool wide_ld(int kind, const GProb& g) {
  const int64_t lim = ((int64_t)1 << 32) / (128 * (kind == 0 ? 8 : 4));
  return std::max(g.lda, g.ldb) >= lim;
}

// The ring tile (k_grouped_ring.h) of a native problem, and the extent of the work
// items its tiles run in: FP64 64x64 and 32x32 tiles share 128x64 items, 3xBF16 ones 64x64.
int ring_of(int kind, int cfg) { return kind == 1 ? (cfg == 1 ? 2 : 0) : (cfg == CFG_WIDE ? 1 : 0); }
int item_rows(int kind, const GProb& g) {
  return kind == 0 && !wide_ld(kind, g) && g.cfg < 2 ? 128 : kind == 2 && g.cfg < 2 ? 64 : CFG_BM[g.cfg];
}
int item_cols(int kind, const GProb& g) { return kind != 1 && !wide_ld(kind, g) && g.cfg < 2 ? 64 : CFG_BN[g.cfg]; }

// The launch of problem g's items.
int launch_of(int kind, const GProb& g) {
  const int combo = 2 * g.ta + g.tb;
  if (g.cfg == CFG_SMALL) return L_OTHER;
  if (wide_ld(kind, g)) return L_WIDE + combo;
  if (kind == 2) return 4 * (g.cfg < 2 ? 3 : g.cfg - CFG_LARGE) + combo;
  return 4 * ring_of(kind, g.cfg) + combo;
}

// Relative duration of one work item of problem g (MFMA work of one k-split of
// one tile, of what reaches into C where the kernel skips the rest, plus a fixed
// epilogue share).
double item_cost(int kind, const GProb& g) {
  const int64_t rows = item_rows(kind, g), cols = item_cols(kind, g);
  const double area = kind == 2 ? (double)(rows * cols) : (double)(std::min(rows, g.m) * std::min(cols, g.n));
  return area * (double)std::max<int64_t>(g.kchunk, 32) + 4096.0;
}

// Resident workgroups per CU of launch L's kernel, from the device's register and
// LDS budget for it (queried once per kernel and device, under the runtime lock;
// the persistent grid is this times the CU count).
hipError_t grouped_occupancy(int kind, int L, int* occ) {
  static int cached[3][NLAUNCH] = {};
  static int cached_device = -1;
  if (cached_device != rt().device) {
    memset(cached, 0, sizeof cached);
    cached_device = rt().device;
  }
  if (cached[kind][L] == 0) {
    const GroupedKernel k = launch_kernel(kind, L);
    int n = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(k.fn), k.threads, 0);
    if (e != hipSuccess) return e;
    cached[kind][L] = std::min(std::max(n, 1), 8);
  }
  *occ = cached[kind][L];
  return hipSuccess;
}

// Workgroups per CU up to which a group is split along k (plan_choices): of the
// 64x64 / 32x32 tiles, and of the 128-row/column tiles, per method kind.  More than
// the MFMA tiles' residency: shorter chains also round less, and these depths are
// the ones the methods' accuracy was measured with.
constexpr int FILL[3][2] = {{4, 2}, {8, 8}, {3, 2}};
// 3xBF16: 64x128 tiles per compute unit from which on each problem takes the tile with the
// least padding.  That is up to four kernels, whose longest items start one kernel after
// the other: 1024 products (17000 tiles) 1378 us with 64x128 tiles, 1253 so; 350 products
// (8524) 525 and 512; 119 (2940) 194 and 218; 53 (1492) 126 and 163.
constexpr int X3_MANY = 32;
// An item longer than this many times a workgroup's share of the group (two per compute
// unit) is split further: it alone would bound the group.  78 FP64 products 431 us without,
// 348 at 1.0 (at 2.0 they are not split); 16 and 31 products in 3xBF16 111 and 99 us
// without, 95.5 and 91 at 2.0, 99 and 101 at 1.0 (26 products 135 at both ends, 143).
constexpr double LONGEST[3] = {1.0, 1.0, 2.0};

// Tile and split of every problem with m, n > 0 (in order), the plan's first
// two passes: the table / tuner / static choice per problem, then the device
// fill: while the group has fewer tiles than FILL workgroups per compute unit (the
// 128-row/column tiles and the others counted apart), the split of its statically
// chosen problem with the longest tiles doubles, down to 256 k per split; then items
// that would bound the group are split (LONGEST).  Last, each split's k range is fixed.  flops: sum of 2 m n k.
int plan_choices(int method, int64_t count, const jb_gemm_desc* d, const Forced& forced, std::vector<GProb>& probs,
                 double* flops) {
  const int kind = kind_of(method);
  std::vector<char> dflt;
  *flops = 0;
  for (int64_t i = 0; i < count; ++i) {
    const jb_gemm_desc& x = d[i];
    if (x.m == 0 || x.n == 0) continue;
    GProb g;
    memset(&g, 0, sizeof g);
    g.A = x.A;
    g.B = x.B;
    g.C = x.C;
    g.m = x.m;
    g.n = x.n;
    g.k = (x.alpha == 0.0) ? 0 : x.k;
    g.lda = x.lda;
    g.ldb = x.ldb;
    g.ldc = x.ldc;
    g.alpha = x.alpha;
    g.beta = x.beta;
    g.ta = !(x.transA == 'N' || x.transA == 'n');
    g.tb = !(x.transB == 'N' || x.transB == 'n');
    bool is_default = false;
    if (forced.cfg >= 0) {
      g.cfg = forced.cfg;
      g.splitk = forced.splitk;
    } else {
      const TuneEntry* o = nullptr;
      if (forced.over) {
        auto it = forced.over->find(bucket_key(method, g.m, g.n, g.k));
        if (it != forced.over->end()) o = &it->second;
      }
      if (o) {
        g.cfg = o->cfg;
        g.splitk = o->splitk;
      } else {
        is_default = choose(method, g.m, g.n, g.k, g.cfg, g.splitk);
      }
    }
    fit_choice(kind, g.m, g.n, g.k, g.cfg, g.splitk);
    if (g.cfg != CFG_SMALL && wide_ld(kind, g)) g.cfg = 0;
    *flops += 2.0 * (double)g.m * (double)g.n * (double)x.k;
    probs.push_back(g);
    dflt.push_back(is_default && g.cfg != CFG_SMALL);
  }
  const int64_t cus = rt().info.compute_units;
  auto tiles = [](const GProb& g) {
    return (g.m + CFG_BM[g.cfg] - 1) / CFG_BM[g.cfg] * ((g.n + CFG_BN[g.cfg] - 1) / CFG_BN[g.cfg]);
  };
  if (kind == 2) {
    int64_t all = 0;
    for (auto& g : probs) all += tiles(g) * std::max(g.splitk, 1);
    for (size_t i = 0; i < probs.size(); ++i)
      if (dflt[i] && all >= X3_MANY * cus && !wide_ld(kind, probs[i])) probs[i].cfg = tile_by_rate(kind, probs[i].m, probs[i].n);
  }
  int64_t items[2] = {0, 0};
  for (auto& g : probs) items[large_cfg(g.cfg)] += tiles(g) * std::max(g.splitk, 1);
  for (;;) {
    int best = -1;
    double best_cost = 0;
    for (size_t i = 0; i < probs.size(); ++i) {
      const GProb& g = probs[i];
      const int q = large_cfg(g.cfg);
      if (!dflt[i] || items[q] >= cus * FILL[kind][q] || g.splitk >= 64 || g.k / (2 * g.splitk) < 256) continue;
      const double cost = (double)CFG_BM[g.cfg] * CFG_BN[g.cfg] * (double)g.k / g.splitk;
      if (cost > best_cost) {
        best_cost = cost;
        best = (int)i;
      }
    }
    if (best < 0) break;
    GProb& g = probs[best];
    items[large_cfg(g.cfg)] += tiles(g) * g.splitk;
    g.splitk *= 2;
  }
  // items that would bound the group
  auto cost = [](const GProb& g) { return (double)CFG_BM[g.cfg] * CFG_BN[g.cfg] * ((double)g.k / g.splitk + 128.0); };
  double total = 0;
  for (auto& g : probs) total += (double)tiles(g) * g.splitk * cost(g);
  for (size_t i = 0; i < probs.size(); ++i) {
    GProb& g = probs[i];
    while (dflt[i] && g.splitk < 64 && g.k / (2 * g.splitk) >= 256 && cost(g) > LONGEST[kind] * total / (2.0 * cus))
      g.splitk *= 2;
  }
  // k per split: a multiple of 32, and no split comes out empty
  for (auto& g : probs) {
    int64_t kc = (g.k + g.splitk - 1) / std::max(g.splitk, 1);
    kc = std::max<int64_t>(32, (kc + 31) / 32 * 32);
    g.splitk = g.k == 0 ? 1 : (int)std::max<int64_t>(1, (g.k + kc - 1) / kc);
    g.kchunk = kc;
    g.tiles_m = (int)((g.m + item_rows(kind, g) - 1) / item_rows(kind, g));
    g.tiles_n = (int)((g.n + item_cols(kind, g) - 1) / item_cols(kind, g));
  }
  return JB_OK;
}

int plan_build(int method, int64_t count, const jb_gemm_desc* d, const Forced& forced, GroupedPlanImpl& P) {
  P.method = method;
  P.kind = kind_of(method);
  const size_t elt = P.kind == 0 ? 8 : 4;
  hipError_t e;
  std::vector<GProb> probs;
  int rc = plan_choices(method, count, d, forced, probs, &P.flops);
  if (rc) return rc;
  // pass 3: arrival counters and partial slabs of the split problems
  size_t part_elems = 0;
  int counters = 0;
  std::vector<size_t> part_off(probs.size(), (size_t)-1);
  std::vector<double> prob_cost(probs.size());
  size_t nall = 0;
  for (size_t pi = 0; pi < probs.size(); ++pi) {
    GProb& g = probs[pi];
    const int ntiles = g.tiles_m * g.tiles_n;
    g.counter_base = counters;
    if (g.splitk > 1) {
      counters += ntiles;
      part_off[pi] = part_elems;
      part_elems += (size_t)ntiles * g.splitk * item_rows(P.kind, g) * item_cols(P.kind, g);
    }
    prob_cost[pi] = item_cost(P.kind, g) * ntiles * g.splitk;
    nall += (size_t)ntiles * g.splitk;
  }
  if (nall >= ((size_t)1 << 31) || (size_t)counters >= ((size_t)1 << 30))
    return fail(JB_ERR_UNSUPPORTED, "grouped plan: %zu work items is too many for one launch", nall);
  // pass 4: work queues.  One launch per kernel (NLAUNCH), each with one queue
  // per XCD.  A problem with at least 2 NXCD items is
  // cut into NXCD runs of consecutive items, one per queue: items are ordered
  // split by split, and within a split tile by tile in groups of `gr`
  // tile-rows (column by column inside a group), so a run is a compact block
  // of tiles sharing A row panels and B column panels.  A smaller problem goes
  // whole to the queue of its launch with the least work so far (problems
  // visited in decreasing order of their work).  Each queue runs its longest
  // items first.
  std::vector<std::pair<double, GItem>> q[NLAUNCH][NXCD];
  double load[NLAUNCH][NXCD] = {};
  std::vector<int> order(probs.size());
  for (size_t i = 0; i < order.size(); ++i) order[i] = (int)i;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return prob_cost[x] > prob_cost[y]; });
  std::vector<GItem> seq;
  for (int pi : order) {
    const GProb& g = probs[pi];
    const int L = launch_of(P.kind, g);
    const int ntiles = g.tiles_m * g.tiles_n;
    const int nitems = ntiles * g.splitk;
    const double c = item_cost(P.kind, g);
    const int per_run = (nitems + NXCD - 1) / NXCD;
    const int gr = std::max(1, std::min(g.tiles_m, (int)std::lround(std::sqrt((double)per_run))));
    seq.clear();
    for (int s2 = 0; s2 < g.splitk; ++s2)
      for (int r0 = 0; r0 < g.tiles_m; r0 += gr)
        for (int tn = 0; tn < g.tiles_n; ++tn)
          for (int tm = r0; tm < std::min(r0 + gr, g.tiles_m); ++tm) seq.push_back(GItem{pi, tm * g.tiles_n + tn, s2, 0});
    if (nitems >= 2 * NXCD) {
      for (int i = 0; i < nitems; ++i) {
        const int x = (int)((int64_t)i * NXCD / nitems);
        q[L][x].push_back({c, seq[i]});
        load[L][x] += c;
      }
    } else {
      int x = 0;
      for (int y = 1; y < NXCD; ++y)
        if (load[L][y] < load[L][x]) x = y;
      for (const GItem& w : seq) q[L][x].push_back({c, w});
      load[L][x] += c * nitems;
    }
  }
  P.nprobs = (int)probs.size();
  P.nitems = (int)nall;
  P.ncounters = NLAUNCH * NXCD + counters;  // queue counters, then per-tile arrival counters
  const size_t ob_probs = 0;
  const size_t ob_items = al256(ob_probs + probs.size() * sizeof(GProb));
  const size_t ob_qdesc = al256(ob_items + nall * sizeof(GItem));
  const size_t ob_cnt = al256(ob_qdesc + (size_t)NLAUNCH * 2 * NXCD * sizeof(int));
  const size_t ob_part = al256(ob_cnt + (size_t)P.ncounters * sizeof(int));
  const size_t total = al256(ob_part + part_elems * elt) + 256;
  const char* fault = getenv("JB_FAULT_ALLOC");
  if (fault && *fault == '1') return fail(JB_ERR_ALLOC, "grouped plan: allocation refused (JB_FAULT_ALLOC)");
  e = hipMalloc(&P.dev, total);
  if (e != hipSuccess) {
    P.dev = nullptr;
    hipGetLastError();
    return fail(JB_ERR_ALLOC, "grouped plan: hipMalloc(%zu) failed: %s", total, hipGetErrorString(e));
  }
  P.dev_bytes = total;
  char* base = static_cast<char*>(P.dev);
  P.probs = reinterpret_cast<GProb*>(base + ob_probs);
  P.items = reinterpret_cast<GItem*>(base + ob_items);
  P.qdesc = reinterpret_cast<int*>(base + ob_qdesc);
  P.next = reinterpret_cast<int*>(base + ob_cnt);
  for (size_t i = 0; i < probs.size(); ++i)
    probs[i].part = part_off[i] == (size_t)-1 ? nullptr : base + ob_part + part_off[i] * elt;
  std::vector<GItem> items;
  std::vector<int> qdesc((size_t)NLAUNCH * 2 * NXCD, 0);
  items.reserve(nall);
  auto by_cost = [](const std::pair<double, GItem>& x, const std::pair<double, GItem>& y) { return x.first > y.first; };
  const int cus = rt().info.compute_units;
  for (int L = 0; L < NLAUNCH; ++L) {
    P.litems[L] = 0;
    for (int x = 0; x < NXCD; ++x) {
      std::stable_sort(q[L][x].begin(), q[L][x].end(), by_cost);
      qdesc[(size_t)L * 2 * NXCD + x] = (int)items.size();
      qdesc[(size_t)L * 2 * NXCD + NXCD + x] = (int)q[L][x].size();
      for (auto& w : q[L][x]) items.push_back(w.second);
      P.litems[L] += (int)q[L][x].size();
    }
    int occ_l = 1;
    if (P.litems[L] > 0 && (e = grouped_occupancy(P.kind, L, &occ_l)) != hipSuccess)
      return hip_fail(e, "grouped plan: occupancy query");
    P.lgrid[L] = std::max(1, std::min(P.litems[L], cus * occ_l));
  }
  if (!probs.empty() && (e = hipMemcpy(P.probs, probs.data(), probs.size() * sizeof(GProb), hipMemcpyHostToDevice)) != hipSuccess)
    return hip_fail(e, "grouped plan: upload problems");
  if (!items.empty() && (e = hipMemcpy(P.items, items.data(), items.size() * sizeof(GItem), hipMemcpyHostToDevice)) != hipSuccess)
    return hip_fail(e, "grouped plan: upload work list");
  if ((e = hipMemcpy(P.qdesc, qdesc.data(), qdesc.size() * sizeof(int), hipMemcpyHostToDevice)) != hipSuccess)
    return hip_fail(e, "grouped plan: upload queue descriptors");
  int nlaunch = 0;
  for (int L = 0; L < NLAUNCH; ++L) nlaunch += P.litems[L] > 0;
  if (log_enabled()) {
    int per_cfg[NCFG] = {}, split = 0;
    for (const GProb& g : probs) {
      ++per_cfg[g.cfg];
      split += g.splitk > 1;
    }
    char launches[256] = "";
    size_t at = 0;
    for (int L = 0; L < NLAUNCH && at < sizeof launches; ++L)
      if (P.litems[L] > 0)
        at += snprintf(launches + at, sizeof launches - at, " [%d: %d items, grid %d]", L, P.litems[L], P.lgrid[L]);
    log_line("grouped plan: method %d, %d problems (64x64 %d, 32x32 %d, small %d, 128x128 %d, 128x64 %d, 64x128 %d;"
             " %d split), %d items, %.4g flops, %zu device bytes, launches%s",
             method, P.nprobs, per_cfg[0], per_cfg[1], per_cfg[2], per_cfg[3], per_cfg[4], per_cfg[5], split,
             P.nitems, P.flops, P.dev_bytes, launches);
  }
  if (nlaunch > 1) {
    if ((e = hipEventCreateWithFlags(&P.fork, hipEventDisableTiming)) != hipSuccess)
      return hip_fail(e, "grouped plan: event");
    for (; P.nside < nlaunch - 1; ++P.nside) {
      if ((e = hipStreamCreateWithFlags(&P.side[P.nside], hipStreamNonBlocking)) != hipSuccess)
        return hip_fail(e, "grouped plan: side stream");
      if ((e = hipEventCreateWithFlags(&P.join[P.nside], hipEventDisableTiming)) != hipSuccess) {
        hipStreamDestroy(P.side[P.nside]);
        P.side[P.nside] = nullptr;
        return hip_fail(e, "grouped plan: event");
      }
    }
  }
  return JB_OK;
}

// Enqueues [reset counters, the launches' persistent kernels (NLAUNCH)] on s and its side streams.
hipError_t plan_enqueue(const GroupedPlanImpl& P, hipStream_t s) {
  if (P.nitems == 0) return hipSuccess;
  hipError_t e = launch_zero_i32(P.next, P.ncounters, s);
  if (e != hipSuccess) return e;
  timing_begin(s, "grouped_gemm");
  if (P.nside > 0 && (e = hipEventRecord(P.fork, s)) != hipSuccess) return e;
  int* const tiles = P.next + NLAUNCH * NXCD;
  int j = -1;  // launch j + 1 > 0 goes to side stream j
  for (int L = 0; L < NLAUNCH; ++L) {
    if (P.litems[L] == 0) continue;
    hipStream_t ls = s;
    if (j >= 0) {
      ls = P.side[j];
      if ((e = hipStreamWaitEvent(ls, P.fork, 0)) != hipSuccess) return e;
    }
    const int* qd = P.qdesc + L * 2 * NXCD;
    int* qn = P.next + L * NXCD;
    const GroupedKernel k = launch_kernel(P.kind, L);
    hipLaunchKernelGGL(k.fn, dim3(P.lgrid[L]), dim3(k.threads), 0, ls, P.probs, P.items, qd, qn, tiles);
    if (j >= 0) {
      if ((e = hipEventRecord(P.join[j], ls)) != hipSuccess) return e;
      if ((e = hipStreamWaitEvent(s, P.join[j], 0)) != hipSuccess) return e;
    }
    ++j;
  }
  timing_end(s, "grouped_gemm");
  return hipGetLastError();
}

void plan_free(GroupedPlanImpl& P) {
  for (int i = 0; i < P.nside; ++i) {
    if (P.side[i]) hipStreamSynchronize(P.side[i]);
    if (P.side[i]) hipStreamDestroy(P.side[i]);
    if (P.join[i]) hipEventDestroy(P.join[i]);
  }
  if (P.fork) hipEventDestroy(P.fork);
  if (P.exec) hipGraphExecDestroy(P.exec);
  if (P.graph) hipGraphDestroy(P.graph);
  if (P.cap) hipStreamDestroy(P.cap);
  if (P.done) hipEventDestroy(P.done);
  if (P.dev) hipFree(P.dev);
  P = GroupedPlanImpl();
}

int plan_capture(GroupedPlanImpl& P) {
  if (getenv("JB_FAULT_GRAPH")) return fail(JB_ERR_GRAPH, "graph capture refused (JB_FAULT_GRAPH)");
  hipError_t e = hipStreamCreateWithFlags(&P.cap, hipStreamNonBlocking);
  if (e != hipSuccess) return hip_fail(e, "grouped plan: capture stream");
  if ((e = hipStreamBeginCapture(P.cap, hipStreamCaptureModeThreadLocal)) != hipSuccess)
    return fail(JB_ERR_GRAPH, "hipStreamBeginCapture: %s", hipGetErrorString(e));
  hipError_t le = plan_enqueue(P, P.cap);
  e = hipStreamEndCapture(P.cap, &P.graph);
  if (le != hipSuccess || e != hipSuccess)
    return fail(JB_ERR_GRAPH, "graph capture failed: %s", hipGetErrorString(le != hipSuccess ? le : e));
  if ((e = hipGraphInstantiate(&P.exec, P.graph, nullptr, nullptr, 0)) != hipSuccess)
    return fail(JB_ERR_GRAPH, "hipGraphInstantiate: %s", hipGetErrorString(e));
  if ((e = hipEventCreateWithFlags(&P.done, hipEventDisableTiming)) != hipSuccess)
    return hip_fail(e, "grouped plan: event");
  return JB_OK;
}

// One-shot grouped launch (no graph), synchronous.
int run_grouped_once(int method, int64_t count, const jb_gemm_desc* d, const Forced& forced, hipStream_t s) {
  GroupedPlanImpl P;
  int rc = plan_build(method, count, d, forced, P);
  if (rc == JB_OK) {
    hipError_t e = plan_enqueue(P, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) rc = hip_fail(e, "grouped launch");
  }
  hipStreamSynchronize(s);
  plan_free(P);
  return rc;
}

}  // namespace

void grouped_release_all() {
  for (auto* p : g_plans) {
    plan_free(p->impl);
    delete p;
  }
  g_plans.clear();
}

// ---- JSON persistence of the table ------------------------------------------
static std::string table_prefix() {
  char buf[160];
  snprintf(buf, sizeof buf, "%s|%s|", rt().info.name, rt().info.arch);
  return buf;
}

int tune_save_locked(const char* path) {
  FILE* f = fopen(path, "w");
  if (!f) return fail(-1, "cannot open %s for writing", path);
  fprintf(f, "{\n  \"format\": \"jblas-tune-1\",\n  \"entries\": [\n");
  size_t i = 0;
  const std::string pre = table_prefix();
  for (auto& kv : g_table) {
    fprintf(f, "    {\"key\": \"%s%s\", \"cfg\": %d, \"splitk\": %d, \"ms\": %.6f}%s\n", pre.c_str(), kv.first.c_str(),
            kv.second.cfg, kv.second.splitk, kv.second.ms, ++i < g_table.size() ? "," : "");
  }
  fprintf(f, "  ]\n}\n");
  fclose(f);
  return JB_OK;
}

int tune_load_locked(const char* path) {
  FILE* f = fopen(path, "r");
  if (!f) return fail(-1, "cannot open %s", path);
  std::string txt;
  char buf[4096];
  size_t nr;
  while ((nr = fread(buf, 1, sizeof buf, f)) > 0) txt.append(buf, nr);
  fclose(f);
  if (txt.find("\"jblas-tune-1\"") == std::string::npos) return fail(JB_ERR_STATE, "%s: not a jblas tuning table", path);
  const std::string pre = table_prefix();
  std::map<std::string, TuneEntry> loaded;
  size_t pos = 0;
  while ((pos = txt.find("{\"key\": \"", pos)) != std::string::npos) {
    pos += 9;
    const size_t q = txt.find('"', pos);
    if (q == std::string::npos) break;
    std::string key = txt.substr(pos, q - pos);
    int cfg = -1, sk = -1;
    double ms = 0;
    if (sscanf(txt.c_str() + q, "\", \"cfg\": %d, \"splitk\": %d, \"ms\": %lf", &cfg, &sk, &ms) != 3)
      return fail(JB_ERR_STATE, "%s: malformed entry", path);
    if (cfg < 0 || cfg >= NCFG || sk < 1 || sk > 64) return fail(JB_ERR_STATE, "%s: entry out of range", path);
    if (key.compare(0, pre.size(), pre) == 0) loaded[key.substr(pre.size())] = TuneEntry{cfg, sk, ms};
    pos = q;
  }
  for (auto& kv : loaded) g_table[kv.first] = kv.second;  // entries of other devices are ignored
  return JB_OK;
}

}  // namespace jb

using namespace jb;

extern "C" {

int jb_gemm_grouped_dev(int method, int64_t count, const jb_gemm_desc* descs, void* stream) {
  int rc = validate_descs(method, count, descs);
  if (rc) return rc;
  std::lock_guard<std::mutex> lk(rt().mu);
  if ((rc = ensure_init())) return rc;
  return run_grouped_once(method, count, descs, Forced(), (hipStream_t)stream);
}

int jb_grouped_plan_create(int method, int64_t count, const jb_gemm_desc* descs, void* stream,
                           jb_grouped_plan** plan) {
  (void)stream;
  if (!plan) return fail(-5, "plan is NULL");
  *plan = nullptr;
  int rc = validate_descs(method, count, descs);
  if (rc) return rc;
  std::lock_guard<std::mutex> lk(rt().mu);
  if ((rc = ensure_init())) return rc;
  auto* p = new jb_grouped_plan();
  rc = plan_build(method, count, descs, Forced(), p->impl);
  if (rc == JB_OK) rc = plan_capture(p->impl);
  if (rc != JB_OK) {
    plan_free(p->impl);
    delete p;
    return rc;
  }
  g_plans.push_back(p);
  *plan = p;
  return JB_OK;
}

int jb_grouped_plan_launch(jb_grouped_plan* plan, void* stream) {
  std::lock_guard<std::mutex> lk(rt().mu);
  if (!plan || std::find(g_plans.begin(), g_plans.end(), plan) == g_plans.end())
    return fail(JB_ERR_STATE, "unknown grouped plan");
  GroupedPlanImpl& P = plan->impl;
  if (P.nitems == 0) return JB_OK;
  hipError_t e = hipSuccess;
  // replays of one plan never overlap: they share its counters
  if (P.launched && (e = hipStreamWaitEvent((hipStream_t)stream, P.done, 0)) != hipSuccess)
    return hip_fail(e, "grouped plan: wait for the previous replay");
  if ((e = hipGraphLaunch(P.exec, (hipStream_t)stream)) != hipSuccess)
    return fail(JB_ERR_GRAPH, "hipGraphLaunch: %s", hipGetErrorString(e));
  if ((e = hipEventRecord(P.done, (hipStream_t)stream)) != hipSuccess) return hip_fail(e, "grouped plan: record replay");
  P.launched = true;
  return JB_OK;
}

int jb_grouped_plan_destroy(jb_grouped_plan* plan) {
  std::lock_guard<std::mutex> lk(rt().mu);
  auto it = std::find(g_plans.begin(), g_plans.end(), plan);
  if (!plan || it == g_plans.end()) return fail(JB_ERR_STATE, "unknown grouped plan");
  hipDeviceSynchronize();
  plan_free(plan->impl);
  delete plan;
  g_plans.erase(it);
  return JB_OK;
}

// Builds the plan of the whole group with the bucket choices `over`, runs it
// once to warm up and `reps` times under events; *ms = the fastest run.
static int autotune_trial(int method, int64_t count, const jb_gemm_desc* descs,
                          const std::map<std::string, TuneEntry>& over, int reps, hipStream_t s, hipEvent_t e0,
                          hipEvent_t e1, double* ms) {
  Forced fc;
  fc.over = &over;
  GroupedPlanImpl P;
  int rc = plan_build(method, count, descs, fc, P);
  if (rc) {
    plan_free(P);
    return rc;
  }
  hipError_t e = plan_enqueue(P, s);
  double best = 1e30;
  for (int r = 0; r < reps && e == hipSuccess; ++r) {
    if ((e = hipEventRecord(e0, s)) != hipSuccess) break;
    if ((e = plan_enqueue(P, s)) != hipSuccess) break;
    if ((e = hipEventRecord(e1, s)) != hipSuccess) break;
    if ((e = hipEventSynchronize(e1)) != hipSuccess) break;
    float t = 0;
    hipEventElapsedTime(&t, e0, e1);
    best = std::min(best, (double)t);
  }
  hipStreamSynchronize(s);
  plan_free(P);
  if (e != hipSuccess) return hip_fail(e, "autotune trial");
  *ms = best;
  return JB_OK;
}

int jb_autotune_grouped(int method, int64_t count, const jb_gemm_desc* descs, int reps, void* stream) {
  int rc = validate_descs(method, count, descs);
  if (rc) return rc;
  if (reps < 1 || reps > 1000) return fail(-4, "reps must be in 1..1000");
  std::lock_guard<std::mutex> lk(rt().mu);
  if ((rc = ensure_init())) return rc;
  hipStream_t s = (hipStream_t)stream;
  // Tuning happens in context: every trial times the whole group, so a
  // bucket's choice is judged by what it does to the group's time (a split-K
  // that helps a bucket alone can slow a group that already fills the GPU).
  // Coordinate descent, one pass, buckets in decreasing order of their flops;
  // a candidate replaces the current choice only if the group gets >= 1 % faster.
  struct Bucket {
    double flops = 0;
    int64_t k = 0;
  };
  std::map<std::string, Bucket> buckets;
  double total = 0;
  for (int64_t i = 0; i < count; ++i) {
    const jb_gemm_desc& d = descs[i];
    if (d.m <= 0 || d.n <= 0 || d.k <= 0) continue;
    Bucket& b = buckets[bucket_key(method, d.m, d.n, d.k)];
    const double f = 2.0 * (double)d.m * (double)d.n * (double)d.k;
    b.flops += f;
    b.k = std::max<int64_t>(b.k, d.k);
    total += f;
  }
  std::vector<std::pair<double, std::string>> order;
  for (auto& kv : buckets)
    if (kv.second.flops >= 0.005 * total) order.push_back({kv.second.flops, kv.first});
  std::sort(order.begin(), order.end(), [](const auto& a, const auto& b) { return a.first > b.first; });
  // Trials write into a zeroed scratch copy of every C (ldc = m): the caller's
  // C is neither read nor written, and beta != 0 problems still read a C.
  const size_t elt = kind_of(method) == 0 ? 8 : 4;
  std::vector<jb_gemm_desc> trial(descs, descs + count);
  size_t cbytes = 0;
  for (auto& d : trial) {
    if (d.m <= 0 || d.n <= 0) continue;
    cbytes = al256(cbytes);
    d.C = reinterpret_cast<void*>(cbytes);  // offset for now
    d.ldc = d.m;
    cbytes += (size_t)d.m * (size_t)d.n * elt;
  }
  void* cscratch = nullptr;
  if (cbytes > 0) {
    const char* fault = getenv("JB_FAULT_ALLOC");
    if (fault && *fault == '1') return fail(JB_ERR_ALLOC, "autotune: allocation refused (JB_FAULT_ALLOC)");
    hipError_t e = hipMalloc(&cscratch, cbytes);
    if (e != hipSuccess) {
      hipGetLastError();
      return fail(JB_ERR_ALLOC, "autotune: hipMalloc(%zu) for the trial outputs failed", cbytes);
    }
    if ((e = hipMemsetAsync(cscratch, 0, cbytes, s)) != hipSuccess) {
      hipFree(cscratch);
      return hip_fail(e, "autotune: clear trial outputs");
    }
    for (auto& d : trial)
      if (d.m > 0 && d.n > 0) d.C = static_cast<char*>(cscratch) + reinterpret_cast<size_t>(d.C);
  }
  descs = trial.data();
  hipEvent_t e0, e1;
  hipEventCreate(&e0);
  hipEventCreate(&e1);
  std::map<std::string, TuneEntry> over;
  double cur = 0;
  // the first trial of a group runs slower (first touch of the operands, clock
  // ramp): a throwaway trial before the baseline keeps the descent from
  // crediting candidates with that difference
  rc = autotune_trial(method, count, descs, over, reps, s, e0, e1, &cur);
  if (rc == JB_OK) rc = autotune_trial(method, count, descs, over, reps, s, e0, e1, &cur);
  for (size_t bi = 0; bi < order.size() && rc == JB_OK; ++bi) {
    const std::string& key = order[bi].second;
    const int64_t kmax = buckets[key].k;
    TuneEntry best{-1, 1, cur};
    for (int cfg = 0; cfg < NCFG && rc == JB_OK; ++cfg)
      for (int sk = 1; sk <= 16 && rc == JB_OK; sk *= 2) {
        if (sk > 1 && kmax / sk < 128) continue;
        if (cfg == CFG_SMALL && (sk > 1 || kmax > SMALL_MAX)) continue;  // one split; k must fit
        if (large_cfg(cfg) && kind_of(method) == 1) continue;               // FP64 and 3xBF16 only
        over[key] = TuneEntry{cfg, sk, 0.0};
        double t = 0;
        rc = autotune_trial(method, count, descs, over, reps, s, e0, e1, &t);
        if (rc == JB_OK && t < 0.99 * best.ms) best = TuneEntry{cfg, sk, t};
      }
    if (best.cfg >= 0) {
      over[key] = best;
      cur = best.ms;
      log_line("autotune %s: tile %d, split %d, group %.4f ms", key.c_str(), best.cfg, best.splitk, best.ms);
    } else {
      over.erase(key);
    }
  }
  // Confirmation: the descent compared single trials, so a choice that only
  // looked >= 1 % faster through timing noise can slip in; the tuned choices
  // are kept only if the whole group, timed again alternately with the
  // static rule (twice as many launches each), is still >= 1 % faster.
  if (rc == JB_OK && !over.empty()) {
    const std::map<std::string, TuneEntry> none;
    double t_static = 1e30, t_tuned = 1e30;
    for (int round = 0; round < 2 && rc == JB_OK; ++round) {
      double t = 0;
      if ((rc = autotune_trial(method, count, descs, none, 2 * reps, s, e0, e1, &t)) != JB_OK) break;
      t_static = std::min(t_static, t);
      if ((rc = autotune_trial(method, count, descs, over, 2 * reps, s, e0, e1, &t)) != JB_OK) break;
      t_tuned = std::min(t_tuned, t);
    }
    if (rc == JB_OK) log_line("autotune confirmation: static %.4f ms, tuned %.4f ms: %s", t_static, t_tuned,
                              t_tuned < 0.99 * t_static ? "kept" : "dropped");
    if (rc == JB_OK && !(t_tuned < 0.99 * t_static)) over.clear();
  }
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  if (cscratch) {
    hipStreamSynchronize(s);
    hipFree(cscratch);
  }
  if (rc) return rc;
  for (auto& kv : over) g_table[kv.first] = kv.second;
  return JB_OK;
}

int jb_autotune_save(const char* path) {
  if (!path) return fail(-1, "path is NULL");
  std::lock_guard<std::mutex> lk(rt().mu);
  int rc = ensure_init();
  if (rc) return rc;
  return tune_save_locked(path);
}

int jb_autotune_load(const char* path) {
  if (!path) return fail(-1, "path is NULL");
  std::lock_guard<std::mutex> lk(rt().mu);
  int rc = ensure_init();
  if (rc) return rc;
  return tune_load_locked(path);
}

int jb_autotune_lookup(int method, int64_t m, int64_t n, int64_t k, int* tile, int* splitk) {
  if (kind_of(method) < 0) return fail(-1, "unknown method");
  if (m < 0 || n < 0 || k < 0) return fail(-2, "negative size");
  if (!tile || !splitk) return fail(-5, "output pointer is NULL");
  std::lock_guard<std::mutex> lk(rt().mu);
  choose(method, m, n, k, *tile, *splitk);
  return JB_OK;
}

int jb_grouped_choices(int method, int64_t count, const jb_gemm_desc* descs, int* tile, int* splitk,
                       int64_t* kchunk) {
  int rc = validate_descs(method, count, descs);
  if (rc) return rc;
  if (count > 0 && (!tile || !splitk || !kchunk)) return fail(-5, "output pointer is NULL");
  std::lock_guard<std::mutex> lk(rt().mu);
  if ((rc = ensure_init())) return rc;
  std::vector<GProb> probs;
  double flops = 0;
  if ((rc = plan_choices(method, count, descs, Forced(), probs, &flops))) return rc;
  size_t j = 0;
  for (int64_t i = 0; i < count; ++i) {
    if (descs[i].m == 0 || descs[i].n == 0) {
      tile[i] = -1;
      splitk[i] = 0;
      kchunk[i] = 0;
      continue;
    }
    tile[i] = probs[j].cfg;
    splitk[i] = probs[j].splitk;
    kchunk[i] = probs[j].kchunk;
    ++j;
  }
  return JB_OK;
}

int jb_autotune_reset(void) {
  std::lock_guard<std::mutex> lk(rt().mu);
  g_table.clear();
  return JB_OK;
}

// ---- pullback -------------------------------------------------------------
static int pullback_descs(char ta, char tb, int64_t m, int64_t n, int64_t k, double alpha, const void* A, int64_t lda,
                          const void* B, int64_t ldb, const void* dC, int64_t lddc, void* dA, int64_t ldda, void* dB,
                          int64_t lddb, std::vector<jb_gemm_desc>& out) {
  const bool tA = !(ta == 'N' || ta == 'n'), tB = !(tb == 'N' || tb == 'n');
  jb_gemm_desc d;
  memset(&d, 0, sizeof d);
  d.alpha = alpha;
  d.beta = 0.0;
  if (dA) {
    // dA (shape of A) = alpha*dC*op(B)^T ('N')  or  alpha*op(B)*dC^T ('T')
    if (!tA) {
      d.transA = 'N'; d.A = dC; d.lda = lddc;
      d.transB = tB ? 'N' : 'T'; d.B = B; d.ldb = ldb;     // op(B)^T
      d.m = m; d.n = k; d.k = n;
    } else {
      d.transA = tB ? 'T' : 'N'; d.A = B; d.lda = ldb;     // op(B)
      d.transB = 'T'; d.B = dC; d.ldb = lddc;              // dC^T
      d.m = k; d.n = m; d.k = n;
    }
    d.C = dA; d.ldc = ldda;
    out.push_back(d);
  }
  if (dB) {
    // dB (shape of B) = alpha*op(A)^T*dC ('N')  or  alpha*dC^T*op(A) ('T')
    if (!tB) {
      d.transA = tA ? 'N' : 'T'; d.A = A; d.lda = lda;     // op(A)^T
      d.transB = 'N'; d.B = dC; d.ldb = lddc;
      d.m = k; d.n = n; d.k = m;
    } else {
      d.transA = 'T'; d.A = dC; d.lda = lddc;              // dC^T
      d.transB = tA ? 'T' : 'N'; d.B = A; d.ldb = lda;     // op(A)
      d.m = n; d.n = k; d.k = m;
    }
    d.C = dB; d.ldc = lddb;
    out.push_back(d);
  }
  return JB_OK;
}

// A large adjoint product fills the GPU on its own; the others (at most two) are split
// along k exactly as a grouped launch of them would be (plan_choices), for the chains
// and the bits of that launch.
static bool pullback_big(const jb_gemm_desc& d) {
  return (double)d.m * (double)d.n >= 256.0 * 128.0 * 128.0 && d.k >= 256;
}

// Every adjoint runs on the single-problem kernels, one after the other on `s`,
// without synchronising.  (The small ones shared a one-shot grouped launch before: its
// lists' allocation and upload, its streams and its synchronisation took 150 us for the
// two products of a 512 x 384 x 256 layer, which take 15 us here.)
static int pullback_run_locked(int method, const std::vector<jb_gemm_desc>& d, hipStream_t s) {
  std::vector<jb_gemm_desc> small;
  for (const jb_gemm_desc& x : d)
    if (x.m > 0 && x.n > 0 && !pullback_big(x)) small.push_back(x);
  std::vector<GProb> probs;
  double flops;
  int rc = small.empty() ? JB_OK : plan_choices(method, (int64_t)small.size(), small.data(), Forced(), probs, &flops);
  if (rc) return rc;
  if (!small.empty() && (rc = refuse_capture(s, "the pullback of a small product"))) return rc;
  auto choice = probs.begin();
  for (const jb_gemm_desc& x : d) {
    if (x.m == 0 || x.n == 0) continue;
    GemmArgs g;
    if ((rc = validate_gemm(x.transA, x.transB, x.m, x.n, x.k, x.alpha == 0.0, x.A, x.lda, x.B, x.ldb, x.C, x.ldc, &g)))
      return rc;
    g.alpha = x.alpha;
    g.beta = x.beta;
    int how = method;
    bool report = true;
    if (!pullback_big(x)) {
      const GProb& c = *choice++;
      if (c.splitk > 1) g.kchunk = c.kchunk;
      if (c.cfg == CFG_SMALL && method == JB_F32_BF16X3) how = JB_F32_NATIVE;  // its FP32 chain
      report = false;
    }
    if ((rc = single_gemm_dev_locked(how, g, s, report))) return rc;
  }
  return JB_OK;
}

static int pullback_validate(int method, char ta, char tb, int64_t m, int64_t n, int64_t k, const void* A, int64_t lda,
                             const void* B, int64_t ldb, const void* dC, int64_t lddc, const void* dA, int64_t ldda,
                             const void* dB, int64_t lddb) {
  if (kind_of(method) < 0) return fail(-1, "method must be JB_F64_NATIVE, JB_F32_NATIVE or JB_F32_BF16X3");
  const bool tA = !(ta == 'N' || ta == 'n'), tB = !(tb == 'N' || tb == 'n');
  if (!(ta == 'N' || ta == 'n' || ta == 'T' || ta == 't' || ta == 'C' || ta == 'c')) return fail(-2, "bad transA");
  if (!(tb == 'N' || tb == 'n' || tb == 'T' || tb == 't' || tb == 'C' || tb == 'c')) return fail(-3, "bad transB");
  if (m < 0) return fail(-4, "m < 0");
  if (n < 0) return fail(-5, "n < 0");
  if (k < 0) return fail(-6, "k < 0");
  const int64_t ar = tA ? k : m, br = tB ? n : k;
  if (dB && m > 0 && !A) return fail(-8, "A is NULL");
  if (lda < std::max<int64_t>(1, ar)) return fail(-9, "lda too small");
  if (dA && n > 0 && !B) return fail(-10, "B is NULL");
  if (ldb < std::max<int64_t>(1, br)) return fail(-11, "ldb too small");
  if (!dC && m > 0 && n > 0) return fail(-12, "dC is NULL");
  if (lddc < std::max<int64_t>(1, m)) return fail(-13, "lddc too small");
  if (dA && ldda < std::max<int64_t>(1, ar)) return fail(-15, "ldda too small");
  if (dB && lddb < std::max<int64_t>(1, br)) return fail(-17, "lddb too small");
  return JB_OK;
}

int jb_gemm_pullback_dev(int method, char transA, char transB, int64_t m, int64_t n, int64_t k, double alpha,
                         const void* A, int64_t lda, const void* B, int64_t ldb, const void* dC, int64_t lddc,
                         void* dA, int64_t ldda, void* dB, int64_t lddb, void* stream) {
  int rc = pullback_validate(method, transA, transB, m, n, k, A, lda, B, ldb, dC, lddc, dA, ldda, dB, lddb);
  if (rc) return rc;
  std::vector<jb_gemm_desc> d;
  pullback_descs(transA, transB, m, n, k, alpha, A, lda, B, ldb, dC, lddc, dA, ldda, dB, lddb, d);
  if (d.empty()) return JB_OK;
  if ((rc = validate_descs(method, (int64_t)d.size(), d.data()))) return rc;
  std::lock_guard<std::mutex> lk(rt().mu);
  if ((rc = ensure_init())) return rc;
  return pullback_run_locked(method, d, (hipStream_t)stream);
}

int jb_gemm_adjoint_dev(int method, char transA, char transB, char transC, int64_t m, int64_t n, int64_t k, double alpha,
                        const void* A, int64_t lda, const void* B, int64_t ldb, const void* dC, int64_t lddc, void* dA,
                        int64_t ldda, void* dB, int64_t lddb, void* stream) {
  const bool tc = !(transC == 'N' || transC == 'n');
  if (!(transC == 'N' || transC == 'n' || transC == 'T' || transC == 't' || transC == 'C' || transC == 'c'))
    return fail(-4, "bad transC");
  // the gradients are those of op(A) and op(B): checked as the outputs of an 'N', 'N' product
  int rc = pullback_validate(method, transA, transB, m, n, k, A, lda, B, ldb, dC, tc ? std::max<int64_t>(1, m) : lddc,
                             nullptr, 1, nullptr, 1);
  if (rc) return rc < -3 ? rc - 1 : rc;
  if (dB && m > 0 && !A) return fail(-9, "A is NULL");
  if (dA && n > 0 && !B) return fail(-11, "B is NULL");
  if (tc && lddc < std::max<int64_t>(1, n)) return fail(-14, "lddc too small");
  if (dA && ldda < std::max<int64_t>(1, m)) return fail(-16, "ldda too small");
  if (dB && lddb < std::max<int64_t>(1, k)) return fail(-18, "lddb too small");
  std::vector<jb_gemm_desc> d;
  pullback_descs('N', 'N', m, n, k, alpha, A, lda, B, ldb, dC, lddc, dA, ldda, dB, lddb, d);
  for (jb_gemm_desc& x : d) {
    // dA = alpha*op(dC)*op(B)^T, dB = alpha*op(A)^T*op(dC)
    const bool tA = !(transA == 'N' || transA == 'n'), tB = !(transB == 'N' || transB == 'n');
    if (x.C == dA) {
      x.transA = tc ? 'T' : 'N';
      x.transB = tB ? 'N' : 'T';
    } else {
      x.transA = tA ? 'N' : 'T';
      x.transB = tc ? 'T' : 'N';
    }
  }
  if (d.empty()) return JB_OK;
  if ((rc = validate_descs(method, (int64_t)d.size(), d.data()))) return rc;
  std::lock_guard<std::mutex> lk(rt().mu);
  if ((rc = ensure_init())) return rc;
  return pullback_run_locked(method, d, (hipStream_t)stream);
}

int jb_gemm_pullback(int method, char transA, char transB, int64_t m, int64_t n, int64_t k, double alpha,
                     const void* A, int64_t lda, const void* B, int64_t ldb, const void* dC, int64_t lddc, void* dA,
                     int64_t ldda, void* dB, int64_t lddb) {
  int rc = pullback_validate(method, transA, transB, m, n, k, A, lda, B, ldb, dC, lddc, dA, ldda, dB, lddb);
  if (rc) return rc;
  const size_t elt = (method == JB_F64_NATIVE) ? 8 : 4;
  const bool tA = !(transA == 'N' || transA == 'n'), tB = !(transB == 'N' || transB == 'n');
  const int64_t ar = tA ? k : m, ac = tA ? m : k, br = tB ? n : k, bc = tB ? k : n;
  // stage host operands in device memory with packed leading dimensions
  std::lock_guard<std::mutex> lk(rt().mu);
  if ((rc = ensure_init())) return rc;
  const size_t sA = al256((size_t)ar * ac * elt), sB = al256((size_t)br * bc * elt), sC = al256((size_t)m * n * elt);
  if ((rc = rt().staging.reserve(2 * (sA + sB) + sC + 256, "staging"))) return rc;
  char* base = static_cast<char*>(rt().staging.ptr);
  char *dAv = base, *dBv = base + sA, *dCv = base + sA + sB, *gA = dCv + sC, *gB = gA + sA;
  hipStream_t s = rt().stream;
  hipError_t e = hipSuccess;
  auto h2d = [&](void* dst, const void* src, int64_t rows, int64_t cols, int64_t ld) {
    if (e == hipSuccess && rows > 0 && cols > 0)
      e = (ld == rows || cols == 1)
              ? hipMemcpyAsync(dst, src, (size_t)rows * cols * elt, hipMemcpyHostToDevice, s)
              : hipMemcpy2DAsync(dst, rows * elt, src, ld * elt, rows * elt, cols, hipMemcpyHostToDevice, s);
  };
  auto d2h = [&](void* dst, const void* src, int64_t rows, int64_t cols, int64_t ld) {
    if (e == hipSuccess && rows > 0 && cols > 0)
      e = (ld == rows || cols == 1)
              ? hipMemcpyAsync(dst, src, (size_t)rows * cols * elt, hipMemcpyDeviceToHost, s)
              : hipMemcpy2DAsync(dst, ld * elt, src, rows * elt, rows * elt, cols, hipMemcpyDeviceToHost, s);
  };
  if (dB) h2d(dAv, A, ar, ac, lda);
  if (dA) h2d(dBv, B, br, bc, ldb);
  h2d(dCv, dC, m, n, lddc);
  if (e != hipSuccess) return hip_fail(e, "pullback: copy to device");
  std::vector<jb_gemm_desc> d;
  pullback_descs(transA, transB, m, n, k, alpha, dAv, std::max<int64_t>(1, ar), dBv, std::max<int64_t>(1, br), dCv,
                 std::max<int64_t>(1, m), dA ? gA : nullptr, std::max<int64_t>(1, ar), dB ? gB : nullptr,
                 std::max<int64_t>(1, br), d);
  if (!d.empty()) {
    rc = validate_descs(method, (int64_t)d.size(), d.data());
    if (rc == JB_OK) rc = pullback_run_locked(method, d, s);
    if (rc) {
      hipStreamSynchronize(s);  // the copies from the caller's memory
      return rc;
    }
  }
  if (dA) d2h(dA, gA, ar, ac, ldda);
  if (dB) d2h(dB, gB, br, bc, lddb);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  return e == hipSuccess ? JB_OK : hip_fail(e, "pullback: copy to host");
}

}  // extern "C"
