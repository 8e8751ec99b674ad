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
#include "jb_internal.h"
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>

namespace jb {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// (1) MFMA GEMM, T = double (v_mfma_f64_16x16x4f64) or float
//     (v_mfma_f32_16x16x4f32).  Both instructions are a sequential fma chain
//     over their four k values in lane-group order (checked on the device bit
//     for bit, denormals and signed zeros included), so with lane group g
//     supplying k = 4t+g every element is one fma chain in increasing k: the
//     jmul! recurrence.
//
//     A block of WGM x WGN waves owns a BTM x BTN tile of C.  Operand stages of
//     BK k stream through an LDS ring of NSLOT slots by direct global->LDS
//     loads, NSLOT - 1 stages ahead, with one barrier per stage and an explicit
//     vmcnt wait for the stage at hand (later stages stay in flight).
//
//     Bound: the matrix cores.  What kept them idle was vector instructions: an
//     MFMA shares the wave's vector issue, and each address add or LDS store in the
//     loop cost more matrix time than its own few cycles (8192^3 FP64 66.6 TF/s with
//     register staging, the same with direct loads and 27 vector instructions per
//     stage, 72.9 with the barrier inside the last MFMA group, 76.3 of 78.6 with
//     none left).  So the loads are buffer loads (descriptor + scalar + lane
//     offset, no arithmetic), the stages are unrolled over the ring (constant LDS
//     offsets), and the next fragments are read behind the first MFMA row of a group.
//     FP64, register-staged form -> this: 1024^3 TN 44.2 -> 35.2 us, 4096^3 64 -> 74
//     TF/s, 2999x1777x2111 on odd leading dimensions 462 -> 382 us; FP32 8192^3 130
//     -> 152 of 157 TF/s.
//
//     LDS images (no padding: the loads write 64 consecutive pieces):
//       rows contiguous (A 'N', B 'T'): [k][R], row r of k-row k at r ^ rswz(k);
//       k contiguous (A 'T', B 'N'):    [R][BK] in 16-byte chunks, chunk c of
//                                       row r at c ^ cswz(r).
//     The XORs spread the 16 rows and 4 k of one fragment read over all 64
//     banks; the loads apply them to the global address of each lane.
//
//     VEC: 16 bytes per lane (16-byte aligned bases, leading dimensions and the
//     contiguous extent multiples of the vector); otherwise 4 bytes per lane,
//     which serves any size and leading dimension through the same LDS image.
//     Rows past the operand read its last row again (those results are not
//     stored).  A last stage shorter than BK reads clamped k, and the
//     fragments replace it: -0.0 from A and +0.0 from B, whose product -0 leaves
//     every chain value unchanged.
// ---------------------------------------------------------------------------
template <typename T> struct Mfma;
template <> struct Mfma<double> {
  typedef d4 acc_t;
  static __device__ __forceinline__ acc_t mma(double x, double y, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, c, 0, 0, 0);
  }
  // Row p of the 16x16 result held in item r of a lane of group g = lane/16.
  static __device__ __forceinline__ int prow(int r, int g) { return 4 * r + g; }
};
template <> struct Mfma<float> {
  typedef f4 acc_t;
  static __device__ __forceinline__ acc_t mma(float x, float y, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int prow(int r, int g) { return 4 * g + r; }
};

// sched_barrier mask: vector and scalar ALU instructions may cross, memory instructions and MFMAs keep their order
constexpr int SCHED_ALU = 6;
#define JB_LDS __attribute__((address_space(3)))
#define JB_INLINE __attribute__((always_inline))  // lambdas of the kernel: never outlined

// One wave's load of 64 x LB bytes into LDS at dst, lane l's from base + so + vo (base and so wave-uniform).
template <int LB>
__device__ __forceinline__ void ring_load(gptr<const void> base, uint32_t vo, uint32_t so, char* dst) {
#ifdef __HIP_DEVICE_COMPILE__  // the descriptor type exists on the device only
  __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(const void*)base, 0, 0xffffffffu, 0x00027000);
  if constexpr (LB == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (JB_LDS void*)dst, 16, vo, so, 0, 0);
  else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (JB_LDS void*)dst, 4, vo, so, 0, 0);
#endif
}

// One operand (R rows of op(A) or columns of op(B)) of the kernel below.
//   RC: element (r, k) at P[r + k*ld], else at P[k + r*ld].
//   WIDE: a lane's byte offset inside a stage may exceed 32 bits.
template <typename T, int R, int BK, bool RC, bool VEC, int NW, bool WIDE>
struct RingOperand {
  static constexpr int EB = sizeof(T);
  static constexpr int LB = VEC ? 16 : 4;                  // bytes per lane of one load
  static constexpr int PB = 64 * LB;                       // bytes per load (one wave)
  static constexpr int BYTES = R * BK * EB;                // one stage
  static constexpr int NP = BYTES / PB / NW;               // loads per wave and stage
  static_assert(NP >= 1 && NP * NW * PB == BYTES, "a stage must split into whole loads per wave");
  static constexpr int ROWB = BK * EB;                     // k contiguous: bytes of one row,
  static constexpr int CPR = ROWB / 16;                    // its 16-byte chunks,
  static constexpr int RPB = ROWB < 256 ? 256 / ROWB : 1;  // and rows per 256 bytes (one pass over the banks)
  static constexpr int EPL = PB / EB;                      // elements per load
  static constexpr int KPL = EPL >= R ? EPL / R : 1;       // rows contiguous: k-rows per load,
  static constexpr int LPK = EPL >= R ? 1 : R / EPL;       // or loads per k-row
  static constexpr int RPL = ROWB <= PB ? PB / ROWB : 0;   // k contiguous: rows per load
  static_assert(RC || RPL >= 1, "a load covers whole rows");
  // The k-rows 4t..4t+3 of one fragment read must start 128 bytes (T = double,
  // two per pass over the banks) or 64 bytes (T = float) apart.
  static __device__ __forceinline__ int rswz(int k) {
    if (EB == 8) return 16 * (k & 1);
    return R >= 64 ? 16 * (k & 3) : 16 * ((k >> 1) & 1);
  }
  static_assert(!RC || R >= 32, "the row swizzle stays inside a k-row");
  static __device__ __forceinline__ int cswz(int r) { return (r / RPB) & (CPR - 1); }

  // LDS element of (r, k); r in [0, R), k in [0, BK)
  static __device__ __forceinline__ int at(int r, int k) {
    if (RC) return k * R + (r ^ rswz(k));
    return r * BK + (((k * EB / 16) ^ cswz(r)) * 16 + (k * EB) % 16) / EB;
  }

  typedef typename std::conditional<WIDE, int64_t, uint32_t>::type Off;
  Off off[NP];  // this lane's byte offset in load i of a stage, from the load's wave-uniform address
  // ld: leading dimension; rmax: last row (vector start) that may be read, relative to the tile's first
  __device__ __forceinline__ void init(int64_t ld, int rmax, int wave, int lane) {
    const int lb = lane * LB;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int p = wave + NW * i;
      if (RC) {
        const int kl = KPL > 1 ? (lb / EB) / R : 0, rl = (lb / EB) % (KPL > 1 ? R : EPL);
        const int r = min(((p % LPK) * EPL + rl) ^ rswz(p * KPL / LPK + kl), rmax);
        off[i] = (Off)r * EB + (Off)kl * (Off)ld * EB + lb % EB;
      } else {
        const int row = p * RPL + lb / ROWB;
        const int k = (((lb % ROWB) / 16 ^ cswz(row)) * 16 + lb % 16) / EB;
        off[i] = (Off)min(row, rmax) * (Off)ld * EB + k * EB + lb % EB;
      }
    }
  }
  // Load i of this wave's share of the stage at k0 into LDS at `dst` (the operand's part of a slot).
  __device__ __forceinline__ void issue(gptr<const T> P, int64_t ld, int64_t k0, int wave, char* dst, int i) const {
    const int p = wave + NW * i;
    const int64_t k = RC ? p * KPL / LPK : 0;  // uniform: first k-row of the load
    if constexpr (WIDE) {
      put((gptr<const char>)(P + (RC ? (k0 + k) * ld : k0)) + off[i], dst + p * PB);
    } else {
      // A buffer load adds the stage's base (descriptor), the load's offset (scalar)
      // and the lane's by itself: no vector address arithmetic is left in the loop
      // (a vector instruction holds up the FP64 matrix pipe).
      ring_load<LB>(P + (RC ? k0 * ld : k0), off[i], (uint32_t)k * (uint32_t)ld * EB, dst + p * PB);
    }
  }
  // The same for the last stage, shorter than BK: k clamped to kmax (last vector start).
  static __device__ __forceinline__ void issue_tail(gptr<const T> P, int64_t ld, int64_t k0, int rmax, int64_t kmax,
                                                    int wave, int lane, char* dst, int i) {
    asm volatile("" : "+v"(lane));  // the addresses are formed here, not ahead of the main loop
    const int p = wave + NW * i, lb = lane * LB;
    gptr<const T> src;
    if (RC) {
      const int kl = KPL > 1 ? (lb / EB) / R : 0, rl = (lb / EB) % (KPL > 1 ? R : EPL);
      const int k = p * KPL / LPK + kl;
      src = P + min(((p % LPK) * EPL + rl) ^ rswz(k), rmax) + min<int64_t>(k0 + k, kmax) * ld;
    } else {
      const int row = p * RPL + lb / ROWB;
      const int k = (((lb % ROWB) / 16 ^ cswz(row)) * 16 + lb % 16) / EB;
      src = P + (int64_t)min(row, rmax) * ld + min<int64_t>(k0 + k, kmax);
    }
    put((gptr<const char>)src + lb % EB, dst + p * PB);
  }
  static __device__ __forceinline__ void put(gptr<const char> src, char* dst) {
    if constexpr (VEC) __builtin_amdgcn_global_load_lds((gptr<const void>)src, (JB_LDS void*)dst, 16, 0, 0);
    else __builtin_amdgcn_global_load_lds((gptr<const void>)src, (JB_LDS void*)dst, 4, 0, 0);
  }
};

// s_waitcnt: at most N vector-memory operations outstanding and every LDS read returned.
template <int N>
__device__ __forceinline__ void wait_ring() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}

template <typename T, bool TA, bool TB, bool VEC, bool WIDE, int BTM, int BTN, int WGM, int WGN, int BK,
          int NSLOT_, int MINW>
__global__ __launch_bounds__(64 * WGM * WGN, MINW) void gemm_mfma_kernel(
    int64_t M, int64_t N, int64_t K, T alpha, const T* __restrict__ A_, int64_t lda, const T* __restrict__ B_, int64_t ldb,
    T beta, T* __restrict__ C, int64_t ldc, int tiles_m, int tiles_n, int acc_from_c) {
  constexpr int NW = WGM * WGN;
  typedef RingOperand<T, BTM, BK, !TA, VEC, NW, WIDE> OA;
  typedef RingOperand<T, BTN, BK, TB, VEC, NW, WIDE> OB;
  constexpr int WIM = BTM / WGM / 16, WIN = BTN / WGN / 16;  // 16 x 16 MFMA blocks per wave along m, n
  constexpr int STAGE_B = OA::BYTES + OB::BYTES;
  constexpr int NLD = OA::NP + OB::NP;  // loads per wave and stage
  constexpr int NSLOT = (NSLOT_ - 2) * NLD < 64 ? NSLOT_ : 63 / NLD + 2;  // the loads a wait leaves in flight fit its counter
  constexpr int VW = VEC ? 16 / (int)sizeof(T) : 1;
  constexpr int NT4 = BK / 4;  // MFMA k-groups per stage
  static_assert(NT4 % 2 == 0, "the fragment buffers alternate over whole stages");
  __shared__ __attribute__((aligned(1024))) char ring[NSLOT * STAGE_B];
  typedef typename Mfma<T>::acc_t acc_t;
  gptr<const T> A = as_global(A_), B = as_global(B_);

  const int nblocks = tiles_m * tiles_n;
  const int tile = xcd_remap(blockIdx.x, nblocks, 8);
  int tm, tn;
  tile_coords(tile, tiles_m, tiles_n, 8, tm, tn);
  const int64_t m0 = (int64_t)tm * BTM, n0 = (int64_t)tn * BTN;

  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int wm0 = (wave % WGM) * (BTM / WGM), wn0 = (wave / WGM) * (BTN / WGN);
  const int g = lane / 16, l16 = lane % 16;

  gptr<const T> At = A + (TA ? m0 * lda : m0), Bt = B + (TB ? n0 : n0 * ldb);
  const int ramax = (int)min<int64_t>(M - m0 - (TA ? 1 : VW), BTM);
  const int rbmax = (int)min<int64_t>(N - n0 - (TB ? VW : 1), BTN);
  const int64_t kamax = K - (TA ? VW : 1), kbmax = K - (TB ? 1 : VW);
  const int nst = (int)((K + BK - 1) / BK);
  const int nfull = (int)(K / BK);
  OA oa;
  OB ob;
  oa.init(lda, ramax, wave, lane);
  ob.init(ldb, rbmax, wave, lane);
  // load i of stage st; tail: the last stage, shorter than BK
  auto issue = [&](int st, int slot, int i, auto tail) JB_INLINE {
    char* dst = ring + slot * STAGE_B;
    const int64_t k0 = (int64_t)st * BK;
    if (decltype(tail)::value) {
      if (i < OA::NP) OA::issue_tail(At, lda, k0, ramax, kamax, wave, lane, dst, i);
      else OB::issue_tail(Bt, ldb, k0, rbmax, kbmax, wave, lane, dst + OA::BYTES, i - OA::NP);
    } else {
      if (i < OA::NP) oa.issue(At, lda, k0, wave, dst, i);
      else ob.issue(Bt, ldb, k0, wave, dst + OA::BYTES, i - OA::NP);
    }
  };

  // Chains start from -0.0: the first MFMA step fma(a, x, -0.0) is then exactly
  // fl(a * x) for every input, the plain first product of the reference
  // recurrence (src/gemm.jl:86), signed zeros included (a start of +0.0 would
  // turn an all -0 chain into +0).  Callers route k == 0 elsewhere.
  // acc_from_c (kernel! semantics, src/kernels.jl:225-233): each chain starts
  // from the element of C instead, every k-step an fma; the caller passes
  // alpha = 1, beta = 0, so the epilogue stores the chain value itself.
  constexpr T acc0 = T(-0.0);
  acc_t acc[WIM][WIN];
#pragma unroll
  for (int i = 0; i < WIM; ++i)
#pragma unroll
    for (int j = 0; j < WIN; ++j) acc[i][j] = acc_t{acc0, acc0, acc0, acc0};
  if (acc_from_c) {
#pragma unroll
    for (int i = 0; i < WIM; ++i) {
      const int64_t m = m0 + wm0 + 16 * i + l16;
#pragma unroll
      for (int j = 0; j < WIN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t n = n0 + wn0 + 16 * j + Mfma<T>::prow(r, g);
          if (m < M && n < N) acc[i][j][r] = C[m + n * ldc];
        }
    }
  }

#pragma unroll
  for (int d = 0; d < NSLOT; ++d)
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      if (d < nfull) issue(d, d, i, std::false_type());
      else if (d < nst) issue(d, d, i, std::true_type());
    }

  T a[2][WIM], b[2][WIN];
  auto frags = [&](int slot, int t, T (&x)[WIM], T (&y)[WIN]) JB_INLINE {
    const T* as = reinterpret_cast<const T*>(ring + slot * STAGE_B);
    const T* bs = reinterpret_cast<const T*>(ring + slot * STAGE_B + OA::BYTES);
#pragma unroll
    for (int i = 0; i < WIM; ++i) x[i] = as[OA::at(wm0 + 16 * i + l16, 4 * t + g)];
#pragma unroll
    for (int j = 0; j < WIN; ++j) y[j] = bs[OB::at(wn0 + 16 * j + l16, 4 * t + g)];
  };
  // Waits for this wave's loads of stage st (all but those of the later stages in
  // flight) and its LDS reads, then for every wave.  A plain barrier: the fence of
  // __syncthreads() would wait for all loads.
  auto arrive = [&](int st, auto steady) JB_INLINE {
    const int later = nst - 1 - st;
    if (decltype(steady)::value || later >= NSLOT - 2) wait_ring<(NSLOT - 2) * NLD>();
    else if (NSLOT >= 4 && later == NSLOT - 3) wait_ring<(NSLOT >= 4 ? NSLOT - 3 : 0) * NLD>();
    else wait_ring<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // Stage st in slot `slot`, whose first fragments are in a[0], b[0].  In its last
  // MFMA group the block meets once: stage st + 1 has landed and every wave has
  // read all of stage st, so its slot takes stage st + NSLOT and the next stage's
  // first fragments are read while that group's MFMAs run.
  // TAIL: the short last stage.  STEADY: stage st + NSLOT is a whole stage.
  auto stage = [&](int st, int slot, int nslot, auto tail, auto steady) JB_INLINE {
    constexpr bool TAIL = decltype(tail)::value, STEADY = decltype(steady)::value;
#pragma unroll
    for (int t = 0; t < NT4; ++t) {
      const int cur = t & 1;
      if (TAIL) {
        const bool past = (int64_t)st * BK + 4 * t + g >= K;
#pragma unroll
        for (int i = 0; i < WIM; ++i) a[cur][i] = past ? T(-0.0) : a[cur][i];
#pragma unroll
        for (int j = 0; j < WIN; ++j) b[cur][j] = past ? T(0.0) : b[cur][j];
      }
      auto ahead = [&]() JB_INLINE {
        if (t + 1 < NT4) {
          frags(slot, t + 1, a[cur ^ 1], b[cur ^ 1]);
        } else if (STEADY || st + 1 < nst) {
          arrive(st + 1, steady);
          frags(nslot, 0, a[cur ^ 1], b[cur ^ 1]);
        }
        __builtin_amdgcn_sched_barrier(SCHED_ALU);
      };
      // The next group's fragments are read behind the first row of MFMAs (whose
      // wait for this group's then covers nothing else).
      if (WIM == 1) ahead();
      // D'[p][q] = sum_k X[p][k] Y[k][q] with X = op(B)^T block (p -> n) and Y = op(A)^T
      // block (q -> m), so a 16-lane group holds 16 consecutive rows of one column of C
      // (coalesced column-major stores).
#pragma unroll
      for (int i = 0; i < WIM; ++i) {
#pragma unroll
        for (int j = 0; j < WIN; ++j) acc[i][j] = Mfma<T>::mma(b[cur][j], a[cur][i], acc[i][j]);
        __builtin_amdgcn_sched_barrier(SCHED_ALU);
        if (i == 0 && WIM > 1) ahead();
        if (t + 1 == NT4) {
          constexpr int PI = (NLD + WIM - 1) / WIM;
#pragma unroll
          for (int q = PI * i; q < PI * (i + 1) && q < NLD; ++q) {
            if (STEADY) issue(st + NSLOT, slot, q, std::false_type());
            else if (!TAIL && st + NSLOT < nfull) issue(st + NSLOT, slot, q, std::false_type());
            else if (!TAIL && st + NSLOT < nst) issue(st + NSLOT, slot, q, std::true_type());
          }
        }
      }
      __builtin_amdgcn_sched_barrier(SCHED_ALU);
    }
  };
  arrive(0, std::false_type());
  frags(0, 0, a[0], b[0]);
  int st = 0, slot = 0, nslot = 1;
  auto next = [&]() JB_INLINE {
    ++st;
    slot = nslot;
    nslot = nslot + 1 == NSLOT ? 0 : nslot + 1;
  };
  // unrolled over the ring, so that every LDS address is a constant offset from a few lane registers
  for (; st + 2 * NSLOT - 1 < nfull; st += NSLOT)
#pragma unroll
    for (int d = 0; d < NSLOT; ++d)
      stage(st + d, d, d + 1 == NSLOT ? 0 : d + 1, std::false_type(), std::true_type());
  for (; st < nfull; next()) stage(st, slot, nslot, std::false_type(), std::false_type());
  if (st < nst) stage(st, slot, nslot, std::true_type(), std::false_type());

  if (m0 + BTM <= M && n0 + BTN <= N) {
    // Interior tile: for each 16-row strip, the beta*C loads are issued
    // together, then the results stored.
#pragma unroll
    for (int i = 0; i < WIM; ++i) {
      T* Ci = C + (m0 + wm0 + 16 * i + l16);
      T cv[WIN][4];
#pragma unroll
      for (int j = 0; j < WIN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          cv[j][r] = beta != T(0) ? Ci[(n0 + wn0 + 16 * j + Mfma<T>::prow(r, g)) * ldc] : T(0);
#pragma unroll
      for (int j = 0; j < WIN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          T c = alpha * acc[i][j][r];
          if (beta != T(0)) c = fma(beta, cv[j][r], c);
          Ci[(n0 + wn0 + 16 * j + Mfma<T>::prow(r, g)) * ldc] = c;
        }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < WIM; ++i) {
    const int64_t m = m0 + wm0 + 16 * i + l16;
#pragma unroll
    for (int j = 0; j < WIN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t n = n0 + wn0 + 16 * j + Mfma<T>::prow(r, g);
        if (m < M && n < N) {
          T c = alpha * acc[i][j][r];
          if (beta != T(0)) c = fma(beta, C[m + n * ldc], c);
          C[m + n * ldc] = c;
        }
      }
  }
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

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

template <typename T, bool WIDE, int BTM, int BTN, int WGM, int WGN, int BK, int NSLOT, int MINW>
static hipError_t launch_gemm_mfma_bt(const GemmArgs& g, hipStream_t s, int acc_from_c) {
  const int tiles_m = (int)((g.m + BTM - 1) / BTM), tiles_n = (int)((g.n + BTN - 1) / BTN);
  const int nblocks = tiles_m * tiles_n;
  // 16-byte loads: aligned bases, and leading dimensions and contiguous extents of whole vectors
  constexpr int VW = 16 / sizeof(T);
  const bool vec = !WIDE && aligned16(g.A) && aligned16(g.B) && g.lda % VW == 0 && g.ldb % VW == 0 &&
                   (g.ta ? g.k : g.m) % VW == 0 && (g.tb ? g.n : g.k) % VW == 0;
  auto A = static_cast<const T*>(g.A);
  auto B = static_cast<const T*>(g.B);
  auto C = static_cast<T*>(g.C);
  const T alpha = (T)g.alpha, beta = (T)g.beta;
  const char* tname = sizeof(T) == 8 ? "dgemm_mfma" : "sgemm_mfma";
#define JB_LAUNCH_V(TA, TB, V)                                                                                          \
  hipLaunchKernelGGL((gemm_mfma_kernel<T, TA, TB, V, WIDE, BTM, BTN, WGM, WGN, BK, NSLOT, MINW>), dim3(nblocks),        \
                     dim3(64 * WGM * WGN), 0, s, g.m, g.n, g.k, alpha, A, g.lda, B, g.ldb, beta, C, g.ldc, tiles_m,     \
                     tiles_n, acc_from_c)
#define JB_LAUNCH(TA, TB)                      \
  do {                                         \
    if (vec) JB_LAUNCH_V(TA, TB, !WIDE);     \
    else JB_LAUNCH_V(TA, TB, false);         \
  } while (0)
  timing_begin(s, tname);
  if (!g.ta && !g.tb) JB_LAUNCH(false, false);
  else if (!g.ta && g.tb) JB_LAUNCH(false, true);
  else if (g.ta && !g.tb) JB_LAUNCH(true, false);
  else JB_LAUNCH(true, true);
#undef JB_LAUNCH_V
#undef JB_LAUNCH
  timing_end(s, tname);
  return hipGetLastError();
}

// Ring configuration <waves along m, along n, k per stage, slots, waves per SIMD> of each tile.  A stage is 16 KB
// (FP64 64-tile) to 32 KB; 128- and 64-tiles keep two slots and several workgroups per CU, whose waves fill each
// other's barriers, the smaller tiles more slots, since their stages are shorter than a load's latency.
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
// Measured, us (128 / 64 / 64x32 / 32): FP64 512^3 63 / 19.0 / 11.7 / 8.1, 1024^3
// 124 / 37.6 / 36.7 / 36.9, 1536^3 178 / 146 / 119 / 119, 3072^3 1023 / 811 / 876 /
// 943, 4096^3 1826 / 1961 / 2038 / 2209; FP32 800x840x900 60 / 20.3 / 20.4 / 18.8,
// 3072^3 519 / 426 / 475 / 526, 4096^3 922 / 986 / 1074 / 1216.
template <typename T>
static hipError_t launch_gemm_mfma(const GemmArgs& g, hipStream_t s, int acc_from_c = 0) {
  constexpr bool F64 = sizeof(T) == 8;
  // A load's offset inside a stage spans up to 128 rows of ld elements (k contiguous) or 32 k of them (rows
  // contiguous).  Past 32 bits (from 2^22 or 2^24 doubles on) the 64x32 tile with 64-bit addresses takes the problem.
  const int64_t lim = ((int64_t)1 << 32) / (int64_t)sizeof(T);
  if (g.lda >= lim / (g.ta ? 128 : 32) || g.ldb >= lim / (g.tb ? 32 : 128))
    return launch_gemm_mfma_bt<T, true, 64, 32, 2, 2, F64 ? 16 : 32, 3, 2>(g, s, acc_from_c);
  // testing: pin one variant ("128", "64", "64x32", "32")
  const char* force = getenv("JB_GEMM_TILE");
  if (force && *force) {
    if (!strcmp(force, "128")) return Ring<T, 128, 128>::run(g, s, acc_from_c);
    if (!strcmp(force, "64")) return Ring<T, 64, 64>::run(g, s, acc_from_c);
    if (!strcmp(force, "64x32")) return Ring<T, 64, 32>::run(g, s, acc_from_c);
    if (!strcmp(force, "32")) return Ring<T, 32, 32>::run(g, s, acc_from_c);
  }
  const int64_t cus = std::max(runtime_compute_units(), 1);
  auto cost = [&](int bm, int bn, double rate, double alone) {
    const int64_t tiles = ((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn);
    const int64_t rounds = (tiles + cus - 1) / cus;
    return (double)(rounds * bm * bn) / (rounds == 1 ? rate * alone : rate);
  };
  const double c128 = cost(128, 128, 1.0, 0.95), c64 = cost(64, 64, F64 ? 0.96 : 0.91, 0.90);
  const double c64x32 = cost(64, 32, F64 ? 0.885 : 0.83, 1.0), c32 = cost(32, 32, F64 ? 0.81 : 0.74, 1.0);
  if (c128 <= std::min(c64, std::min(c64x32, c32))) return Ring<T, 128, 128>::run(g, s, acc_from_c);
  if (c64 <= std::min(c64x32, c32)) return Ring<T, 64, 64>::run(g, s, acc_from_c);
  return c64x32 < c32 ? Ring<T, 64, 32>::run(g, s, acc_from_c) : Ring<T, 32, 32>::run(g, s, acc_from_c);
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
