// k_grouped_x3.hip -- persistent kernels of the grouped 3xBF16 method's MFMA tiles.
#include <type_traits>

#include "jb_grouped.h"

namespace jb {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
#define JB_INLINE __attribute__((always_inline))  // lambdas of the kernels: never outlined

// LDS rows of the 3xBF16 tile hold BK = 32 BF16 (64 bytes, four 16-byte chunks,
// no padding); chunk c of row r is stored at chunk c ^ ((r >> 2) & 3), so the 16
// rows that one 16-byte fragment read covers (same c) hit 16 distinct 4-bank
// groups of the 64-bank LDS.
__device__ __forceinline__ int bf_chunk(int r, int c) { return c ^ ((r >> 2) & 3); }

// One operand's stages (R rows x 32 k): raw FP32 runs of four k of one row in registers,
// loaded through a buffer descriptor (the stage's base in scalar registers, one lane
// offset per run; WIDE: 64-bit offsets), then split plane by plane into LDS.  A run of
// a k-contiguous operand is one 16-byte load, which needs 4-byte alignment only.
//   RC (rows contiguous): run q of thread t is row t % R, k-run t / R + (NTH / R) q
//   otherwise:            row t / 8 + (NTH / 8) q, k-run t % 8
// Lanes with consecutive t take consecutive addresses of the contiguous index.  Rows
// past the operand read its last row: they meet only rows or columns outside C.
template <int R, bool RC, bool WIDE, int NTH>
struct XRuns {
  static constexpr int BK = 32, NR = R * BK / (4 * NTH);
  static_assert(R * BK == 4 * NTH * NR && (!RC || NTH % R == 0), "run map");
  typedef float V4 __attribute__((ext_vector_type(4)));
  V4 v[NR];
  typename std::conditional<WIDE, int64_t, uint32_t>::type vo[NR];  // bytes from the stage's base
  uint32_t wo[NR];  // LDS bytes of the run in plane 0
  __device__ __forceinline__ static int row(int t, int q) { return RC ? t % R : t / (BK / 4) + (4 * NTH / BK) * q; }
  __device__ __forceinline__ static int krun(int t, int q) { return RC ? t / R + (NTH / R) * q : t % (BK / 4); }
  __device__ __forceinline__ void begin(int t, int64_t ld, int64_t rows) {
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      const int r = row(t, q), k = krun(t, q);
      const int64_t rc = r < rows ? r : rows - 1;
      vo[q] = (decltype(vo[0] + 0))(4 * (RC ? rc + 4 * k * ld : rc * ld + 4 * k));
      wo[q] = 2 * (r * BK + 8 * bf_chunk(r, k >> 1) + 4 * (k & 1));
    }
  }
  // Run q of the stage at `base`, with nk k left (the last stage may have fewer than 32).
  // From `records` bytes on, past the operand's last element, the buffer load reads zeros
  // (checked per 4 bytes), so a rows-contiguous operand is zero from k = nk on.
  __device__ __forceinline__ void load(int t, int q, gptr<const float> base, uint32_t records, int64_t ld, int nk) {
    if constexpr (WIDE) {
      const int k = 4 * krun(t, q);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[q][e] = k + e < nk ? *(gptr<const float>)((gptr<const char>)base + vo[q] + 4 * e * (RC ? ld : 1)) : 0.0f;
    } else {
#ifdef __HIP_DEVICE_COMPILE__
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          (void*)base, 0, records, 0x00027000);
      if constexpr (!RC) {
        v[q] = __builtin_bit_cast(V4, __builtin_amdgcn_raw_buffer_load_b128(rs, vo[q], 0, 0));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[q][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, vo[q], 4 * e * (uint32_t)ld, 0));
      }
#endif
    }
  }
  // k from nk on of a k-contiguous run, which the load took from the next row
  __device__ __forceinline__ void mask(int t, int q, int nk) {
    if (RC || WIDE) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[q][e] = 4 * krun(t, q) + e < nk ? v[q][e] : 0.0f;
  }
  // plane p of run q, in order 0, 1, 2: x = hi + mid + lo + rest, each plane x rounded to
  // BF16 (nearest even) and subtracted exactly before the next.  |x| within half a BF16
  // ulp of FLT_MAX rounds to Inf: the first plane rounds x clamped to the largest finite
  // BF16, which for such an x is its truncation (the residual then has at most 16
  // significant bits and the split stays exact, as in the single-problem split) and for
  // every other finite x changes nothing.  An Inf or NaN x still leaves a NaN residual,
  // so every product it enters is NaN.
  __device__ __forceinline__ void plane(int q, int p, char* S) {
    V4& x = v[q];
    float y[4] = {x[0], x[1], x[2], x[3]};
    if (p == 0) {
      const float BMAX = __uint_as_float(0x7F7F0000u);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = __builtin_amdgcn_fmed3f(x[e], -BMAX, BMAX);
    }
    const uint32_t w0 = __builtin_bit_cast(uint32_t, bf2{(__bf16)y[0], (__bf16)y[1]});
    const uint32_t w1 = __builtin_bit_cast(uint32_t, bf2{(__bf16)y[2], (__bf16)y[3]});
    *reinterpret_cast<uint2*>(S + wo[q] + p * (R * BK * 2)) = uint2{w0, w1};
    if (p < 2) {
      // x minus its rounding as a dot product of the packed pair with (-1, 0) or (0, -1):
      // one instruction in place of an unpacking shift or mask and a subtraction, with the
      // same result for every input (checked on the device bit for bit, denormals, signed
      // zeros, infinities and the largest values included; a NaN spreads to the other k of
      // its pair, which feeds the same results).  The register constant: as an inline
      // constant -1.0 stands for (0, -1).
      uint32_t lo = 0x0000bf80u;
      asm("" : "+s"(lo));
      const bf2 first = __builtin_bit_cast(bf2, lo), second = __builtin_bit_cast(bf2, 0xbf800000u);
#ifdef __HIP_DEVICE_COMPILE__
      x[0] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, w0), first, x[0], false);
      x[1] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, w0), second, x[1], false);
      x[2] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, w1), first, x[2], false);
      x[3] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, w1), second, x[3], false);
#endif
    }
  }
};

// One work item's stages: WM x WN waves of (BM/WM) x (BN/WN), each a grid of 32x32
// blocks of v_mfma_f32_32x32x16_bf16.  LDS: two stages of [plane][row][32 k], chunks
// swizzled by bf_chunk; a fragment of k-step h is chunk 2h + lane/32 of row lane%32.
// Products t + u <= 4 of the planes, the first in one accumulator, the rest in another.
// Bound: the split's vector instructions beside the products (150 to 220 a stage and
// wave, 24 MFMAs of 32 cycles).  So a stage is one basic block in which the next stage's
// split runs between the MFMAs, a plane of a run at a time, and each run is reloaded as
// soon as it is split: all waves of a SIMD otherwise did their MFMAs together and then
// their splits together.  64 products of 1024^3, k-contiguous operands: 128x128 tile 158
// TF/s so, 173 here (1040 of BF16 products), 64x64 23 (guarded element loads, split
// after the MFMAs) and 143; 1021 x 1021 x 1023: 146 and 165 (128x128).  1024 uneven
// products in one plan: 1465 us, 1378 with the 128-row/column tiles so, 1326 with the
// 64x64 kernel and the choice of tiles by padding, 1309 with the residuals by dot
// products, 1203 with the record counts out of the loop (a 64-bit compare per load of a
// stage: a vector instruction and a wait for its scalar result).
template <int BM, int BN, int WM, int WN, bool TA, bool TB, bool WIDE>
__device__ __forceinline__ void x3_loop(const GProb& P, int64_t m0, int64_t n0, int64_t kb, int64_t ke, char* smem,
                                              f16v (&acc)[2][BM / WM / 32][BN / WN / 32]) {
  constexpr int NTH = 64 * WM * WN, BK = 32;
  constexpr int IB = BM / WM / 32, JB = BN / WN / 32, NB = IB * JB;  // 32x32 blocks per wave
  constexpr int AB = 3 * BM * BK * 2, BUF = AB + 3 * BN * BK * 2;    // bytes of A's planes, of a stage
  typedef XRuns<BM, !TA, WIDE, NTH> RA;
  typedef XRuns<BN, TB, WIDE, NTH> RB;
  const int tid = work_item_tid();
  const int lane = tid % 64, wave = tid / 64;
  const int l32 = lane % 32, hl = lane / 32;
  const int64_t lda = P.lda, ldb = P.ldb;
  gptr<const float> A = as_global(static_cast<const float*>(P.A)) + (TA ? kb + m0 * lda : m0 + kb * lda);
  gptr<const float> B = as_global(static_cast<const float*>(P.B)) + (TB ? n0 + kb * ldb : kb + n0 * ldb);
  const int64_t sa = TA ? BK : BK * lda, sb = TB ? BK * ldb : BK;  // from stage to stage
  RA ra;
  RB rb;
  ra.begin(tid, lda, P.m - m0);
  rb.begin(tid, ldb, P.n - n0);
  const int K = (int)(ke - kb), nkt = (K + BK - 1) / BK;
  // bytes from the last stage's base to the operand's end (earlier stages' loads end inside it)
  const int kl = K - (nkt - 1) * BK;
  const uint32_t reca = buffer_records<float>(TA ? (P.m - m0 - 1) * lda + kl : (kl - 1) * lda + P.m - m0);
  const uint32_t recb = buffer_records<float>(TB ? (kl - 1) * ldb + P.n - n0 : (P.n - n0 - 1) * ldb + kl);
  auto load = [&](int kt, int q) JB_INLINE {
    const bool last = kt == nkt - 1;
    if (q < RA::NR) ra.load(tid, q, A + kt * sa, last ? reca : 0xffffffffu, lda, K - kt * BK);
    else rb.load(tid, q - RA::NR, B + kt * sb, last ? recb : 0xffffffffu, ldb, K - kt * BK);
  };
  auto mask = [&](int kt, int q) JB_INLINE {
    if (q < RA::NR) ra.mask(tid, q, K - kt * BK);
    else rb.mask(tid, q - RA::NR, K - kt * BK);
  };
  // fragment addresses: the two k-steps' chunks differ by an exclusive or with 2
  const int ar = (wave % WM) * (BM / WM) + l32, br = (wave / WM) * (BN / WN) + l32;
  const uint32_t fa[2] = {2u * (ar * BK + 8 * bf_chunk(ar, hl)), 2u * (ar * BK + 8 * bf_chunk(ar, 2 + hl))};
  const uint32_t fb[2] = {AB + 2u * (br * BK + 8 * bf_chunk(br, hl)), AB + 2u * (br * BK + 8 * bf_chunk(br, 2 + hl))};
  bf8 a[2][3][IB], b[2][3][JB];
  // fragment f of k-step h, in the order the products need them: planes 0 of A and B first
  constexpr int NF = 3 * (IB + JB);
  auto frag = [&](const int h, const int f, const char* S) JB_INLINE {
    const int p = f / (IB + JB), i = f % (IB + JB);
    if (i < IB) a[h][p][i] = *reinterpret_cast<const bf8*>(S + fa[h] + (p * BM + 32 * i) * BK * 2);
    else b[h][p][i - IB] = *reinterpret_cast<const bf8*>(S + fb[h] + (p * BN + 32 * (i - IB)) * BK * 2);
  };
  // product x of 6 of every block: X = op(B) plane (p -> n), Y = op(A) plane (q -> m)
  auto mfma = [&](const int h, const int x, const int blk) JB_INLINE {
    constexpr int PB[6] = {0, 1, 0, 2, 1, 0}, PA[6] = {0, 0, 1, 0, 1, 2};
    const int i = blk / JB, j = blk % JB, l = x > 0;
    acc[l][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[h][PB[x]][j], a[h][PA[x]][i], acc[l][i][j], 0, 0, 0);
  };
  constexpr int NM = 12 * NB, NP = 3 * (RA::NR + RB::NR);  // MFMAs and split pieces of a stage
  // One stage.  split: stage kt + 1 from the runs to the other buffer (2: the last stage,
  // past whose end k is masked); reload: stage kt + 2 into the runs.
  auto stage = [&](const int kt, auto split, auto reload) JB_INLINE {
    const char* S = smem + (kt & 1) * BUF;
    char* D = smem + (~kt & 1) * BUF;
#pragma unroll
    for (int f = 0; f < NF; ++f) frag(0, f, S);
#pragma unroll
    for (int x = 0; x < NM; ++x) {
      __builtin_amdgcn_sched_barrier(0);
      const int h = x / (6 * NB);
      mfma(h, x % (6 * NB) / NB, x % NB);
      if (x < NF) frag(1, x, S);
      if constexpr (NM / 2 < NF) {
        if (x == NM / 2 - 1)
#pragma unroll
          for (int f = NM / 2; f < NF; ++f) frag(1, f, S);
      }
      if constexpr (decltype(split)::value > 0) {
#pragma unroll
        for (int y = x * NP / NM; y < (x + 1) * NP / NM; ++y) {
          const int q = y / 3, p = y % 3;
          if (decltype(split)::value == 2 && p == 0) mask(kt + 1, q);
          if (q < RA::NR) ra.plane(q, p, D);
          else rb.plane(q - RA::NR, p, D + AB);
          if (decltype(reload)::value && p == 2) load(kt + 2, q);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (decltype(split)::value > 0) __syncthreads();
  };
  constexpr int NR = RA::NR + RB::NR;
#pragma unroll
  for (int q = 0; q < NR; ++q) load(0, q);
#pragma unroll
  for (int q = 0; q < NR; ++q) {
    mask(0, q);
#pragma unroll
    for (int p = 0; p < 3; ++p)
      if (q < RA::NR) ra.plane(q, p, smem);
      else rb.plane(q - RA::NR, p, smem + AB);
  }
  if (nkt > 1) {
#pragma unroll
    for (int q = 0; q < NR; ++q) load(1, q);
  }
  __syncthreads();
  int kt = 0;
#pragma unroll 1
  for (; kt + 2 < nkt; ++kt) stage(kt, std::integral_constant<int, 1>(), std::true_type());
  if (kt + 1 < nkt) {
    stage(kt, std::integral_constant<int, 2>(), std::false_type());
    ++kt;
  }
  stage(kt, std::integral_constant<int, 0>(), std::false_type());
}

template <int BM, int BN, int WM, int WN, bool TA, bool TB, bool WIDE>
__device__ void x3_tile(const GProb& P, int tm, int tn, int split, char* smem, int* counters, int* sflag) {
  constexpr int NTH = 64 * WM * WN;
  constexpr int IB = BM / WM / 32, JB = BN / WN / 32;
  static_assert(IB >= 1 && JB >= 1 && IB * WM * 32 == BM && JB * WN * 32 == BN, "wave grid");
  const int tid = work_item_tid();
  const int lane = tid % 64, wave = tid / 64;
  const int wm0 = (wave % WM) * (BM / WM), wn0 = (wave / WM) * (BN / WN);
  const int l32 = lane % 32, hl = lane / 32;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int64_t kb = (int64_t)split * P.kchunk;
  const int64_t ke = min(P.k, kb + P.kchunk);
  f16v acc[2][IB][JB];
#pragma unroll
  for (int l = 0; l < 2; ++l)
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
      for (int j = 0; j < JB; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[l][i][j][e] = 0.0f;
  if (kb < ke) x3_loop<BM, BN, WM, WN, TA, TB, WIDE>(P, m0, n0, kb, ke, smem, acc);
  // item e of lane l in block (i, j): row wm0 + 32 i + l%32, column wn0 + 32 j + 8 (e/4) + 4 (l/32) + e%4
  if (!WIDE && P.splitk == 1 && kb < ke && (float)P.beta == 0.0f && P.ldc < (1 << 22)) {
#ifdef __HIP_DEVICE_COMPILE__
    // One multiply and one buffer store per element: columns in scalar offsets, rows in the
    // lane's; columns past C lie past the record count, where stores are dropped.  (The
    // general form below forms and checks an address per element: 1024 uneven products
    // 1228 us, 1197 so; groups of 20 to 700 products 4.6 to 8.4 % faster.)
    const int rows = (int)min<int64_t>(P.m - m0, BM), cols = (int)min<int64_t>(P.n - n0, BN);
    const uint32_t ld = 4 * (uint32_t)P.ldc;
    gptr<float> C = as_global(static_cast<float*>(P.C)) + m0 + n0 * P.ldc;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)C, 0, buffer_records<float>((cols - 1) * P.ldc + rows), 0x00027000);
    const float alpha = (float)P.alpha;
#pragma unroll
    for (int i = 0; i < IB; ++i) {
      const int r = wm0 + 32 * i + l32;
      const uint32_t vo = 4 * (uint32_t)r + (uint32_t)(wn0 + 4 * hl) * ld;
      if (r < rows) {
#pragma unroll
        for (int j = 0; j < JB; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(alpha * (acc[0][i][j][e] + acc[1][i][j][e])), rs, vo,
                                                  (32 * j + 8 * (e / 4) + e % 4) * ld, 0);
      }
    }
#endif
    return;
  }
#pragma unroll
  for (int i = 0; i < IB; ++i)
#pragma unroll
    for (int j = 0; j < JB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        put_result<float, BM, BN>(P, tm, tn, split, wm0 + 32 * i + l32, wn0 + 32 * j + 8 * (e / 4) + 4 * hl + e % 4,
                                  acc[0][i][j][e] + acc[1][i][j][e]);
  splitk_combine<float, BM, NTH>(P, tm, tn, BN, counters, sflag);
}

// Pulls items of one tile shape and transpose combination from their queues.  128x64
// and 64x128: four waves of 64x32 / 32x64, 72 KB (two workgroups per CU); 128x128:
// eight waves of 64x32, 96 KB (one); 64x64: four waves of 32x32, 48 KB (three).
template <int BM, int BN, bool TA, bool TB, bool WIDE>
struct X3Kernel {
  static constexpr int WM = 2, WN = (BM == 128 && BN == 128) ? 4 : 2;
  static constexpr int NTH = 64 * WM * WN;
  static constexpr int MINB = BM + BN == 256 ? 1 : BM + BN == 128 && !WIDE ? 3 : 2;  // workgroups per CU for the register budget
};
template <int BM, int BN, bool TA, bool TB, bool WIDE>
__global__ __launch_bounds__((X3Kernel<BM, BN, TA, TB, WIDE>::NTH), (X3Kernel<BM, BN, TA, TB, WIDE>::MINB))
void grouped_x3_kernel(const GProb* __restrict__ probs, const GItem* __restrict__ items,
                             const int* __restrict__ qdesc, int* __restrict__ qnext, int* __restrict__ counters) {
  typedef X3Kernel<BM, BN, TA, TB, WIDE> K;
  constexpr int SMEM = 2 * 3 * (BM + BN) * 32 * 2;
  __shared__ __attribute__((aligned(16))) char smem[SMEM];
  __shared__ int s_item, s_flag;
  int q = blockIdx.x % NXCD, tries = 0;
  for (;;) {
    const int it = pop_item(qdesc, qnext, q, tries, &s_item);
    if (it < 0) break;
    const GItem w = items[it];
    const GProb P = probs[w.prob];
    const int tm = w.tile / P.tiles_n, tn = w.tile % P.tiles_n;
    x3_tile<BM, BN, K::WM, K::WN, TA, TB, WIDE>(P, tm, tn, w.split, smem, counters, &s_flag);
  }
}

template <int BM, int BN, bool WIDE>
GroupedKernel x3_kernel_of(int combo) {
  static const GroupedKernelFn fn[4] = {
      grouped_x3_kernel<BM, BN, false, false, WIDE>, grouped_x3_kernel<BM, BN, false, true, WIDE>,
      grouped_x3_kernel<BM, BN, true, false, WIDE>, grouped_x3_kernel<BM, BN, true, true, WIDE>};
  return {fn[combo], X3Kernel<BM, BN, false, false, WIDE>::NTH};
}

}  // namespace

GroupedKernel grouped_x3(int which, int combo) {
  switch (which) {
    case 0: return x3_kernel_of<128, 128, false>(combo);
    case 1: return x3_kernel_of<128, 64, false>(combo);
    case 2: return x3_kernel_of<64, 128, false>(combo);
    default: return x3_kernel_of<64, 64, false>(combo);
  }
}
GroupedKernelFn grouped_x3_wide_ld(int combo) { return x3_kernel_of<64, 64, true>(combo).fn; }

}  // namespace jb
