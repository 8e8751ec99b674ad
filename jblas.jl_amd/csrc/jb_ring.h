// jb_ring.h -- the MFMA GEMM tile of the native FP64 and FP32 kernels (the
// single-problem GEMM, k_dgemm.hip, and the grouped launches, k_grouped_ring.hip).
#pragma once
#include <type_traits>

#include "jb_internal.h"

namespace jb {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// MFMA tile, T = double (v_mfma_f64_16x16x4f64) or float
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
//     FP64, register-staged form -> this: 1024^3 TN 44.2 -> 35.2 us, 4096^3 64 -> 76
//     TF/s, 2999x1777x2111 on odd leading dimensions 462 -> 359 us; FP32 8192^3 130
//     -> 152 of 157 TF/s.
//
//     A short product's time is the prologue and the first stages: loads issued one by
//     one behind vector arithmetic on uniform values, descriptors that had become vector
//     values (a loop per load) and stages on run-time slots took 64^3 FP64 from 3.4 us
//     (register-staged) to 4.0, 96^3 TN 3.9 to 4.9; scalar throughout and with the last
//     stages unrolled 3.2 and 3.8, 256^3 6.4 -> 5.8 -> 5.1, FP32 256^3 9.2 -> 5.4 -> 4.7.
//
//     LDS images (no padding: the loads write 64 consecutive pieces):
//       rows contiguous (A 'N', B 'T'): [k][R], row r of k-row k at r ^ rswz(k);
//       k contiguous (A 'T', B 'N'):    [R][BK] in 16-byte chunks, chunk c of
//                                       row r at c ^ cswz(r).
//     The XORs spread the 16 rows and 4 k of one fragment read over all 64
//     banks; the loads apply them to the global address of each lane.
//
//     16 bytes per lane, whatever the sizes and leading dimensions: a buffer load needs
//     4-byte alignment only.  A vector that starts inside the contiguous extent may end
//     past it: in the next column's elements, or, at the end of the operand, past the
//     descriptor's record count, where the load returns zeros (checked per 4 bytes).
//     Every stage that can reach the operand's end has that count (RingOperand::REACH).
//     What it brings there is not used: rows past the operand feed results that are
//     not stored (vectors wholly past it read its last one again), and a last stage
//     shorter than BK, whose later vectors read clamped k, has its fragments past the
//     last k replaced: -0.0 from A and +0.0 from B, whose product -0 leaves every chain
//     value unchanged.  (Odd sizes took 4-byte loads before:
//     2999x1777x2111 FP64 on odd leading dimensions 382 us, 359 so; 209 uneven FP32
//     products of odd sizes in one plan 430 and 410.)
//     WIDE: 4 bytes per lane and 64-bit addresses, every element clamped on its own.
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

// One wave's load of 64 x 16 bytes into LDS at dst, lane l's from base + so + vo (base and so wave-uniform);
// zeros from `records` bytes after base on.
__device__ __forceinline__ void ring_load(gptr<const void> base, uint32_t records, uint32_t vo, uint32_t so, char* dst) {
#ifdef __HIP_DEVICE_COMPILE__  // the descriptor type exists on the device only
  __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(const void*)base, 0,
                                                                  __builtin_amdgcn_readfirstlane(records), 0x00027000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (JB_LDS void*)dst, 16, vo, so, 0, 0);
#endif
}

// One operand (R rows of op(A) or columns of op(B)) of the kernel below.
//   RC: element (r, k) at P[r + k*ld], else at P[k + r*ld].
//   WIDE: a lane's byte offset inside a stage may exceed 32 bits.
// The address functions are host functions too: their bounds are checked there.
#define JB_HD __host__ __device__ __forceinline__
template <typename T, int R, int BK, bool RC, int NW, bool WIDE>
struct RingOperand {
  static constexpr int EB = sizeof(T);
  static constexpr int LB = WIDE ? 4 : 16;                 // bytes per lane of one load
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
  static JB_HD int rswz(int k) {
    if (EB == 8) return 16 * (k & 1);
    return R >= 64 ? 16 * (k & 3) : 16 * ((k >> 1) & 1);
  }
  static_assert(!RC || R >= 32, "the row swizzle stays inside a k-row");
  static JB_HD int cswz(int r) { return (r / RPB) & (CPR - 1); }

  // LDS element of (r, k); r in [0, R), k in [0, BK)
  static JB_HD int at(int r, int k) {
    if (RC) return k * R + (r ^ rswz(k));
    return r * BK + (((k * EB / 16) ^ cswz(r)) * 16 + (k * EB) % 16) / EB;
  }

  typedef typename std::conditional<WIDE, int64_t, uint32_t>::type Off;
  Off off[NP];  // this lane's byte offset in load i of a stage, from the load's wave-uniform address
  // ld: leading dimension; rmax: last row (vector start) that may be read, relative to the tile's first
  JB_HD void init(int64_t ld, int rmax, int wave, int lane) {
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

  // Whether a vector of the stage before the last can end past the operand: with more than two elements to a vector
  // and ld below its length, it runs over the few elements of a short last stage (one row of ld 1, K = 33: the vector
  // at k = 31 covers k = 31..34).  Earlier stages have a whole one after them; k-contiguous ones end with their k.
  static constexpr bool REACH = RC && 16 / EB > 2;
  // elements from a stage's base to the operand's end, kleft k from the stage's first on
  static JB_HD int64_t extent(int64_t ld, int64_t rows, int64_t kleft) {
    return RC ? (kleft - 1) * ld + rows : (rows - 1) * ld + kleft;
  }
  // First k-row of load p of a stage (uniform).  TAIL: the last stage, shorter than BK, whose last vectors start at kleft.
  template <bool TAIL>
  static JB_HD int krow(int p, int kleft) {
    return RC ? (TAIL ? min(p * KPL / LPK, kleft) : p * KPL / LPK) : 0;
  }
  // Bytes by which this lane's vector of such a stage's load p (first k-row kp) starts past kleft.
  static JB_HD Off past(int p, int kp, int kleft, int64_t ld, int lane) {
    const int lb = lane * LB;
    if (RC) return KPL > 1 ? (Off)max((lb / EB) / R - (kleft - kp), 0) * (Off)ld * EB : 0;
    const int k = (((lb % ROWB) / 16 ^ cswz(p * RPL + lb / ROWB)) * 16 + lb % 16) / EB;
    return (Off)max(k - kleft, 0) * EB;
  }
  // Load i of this wave's share of the stage at k0 into LDS at `dst` (the operand's part of a slot).  P: the operand
  // at the tile's first row.  TAIL: the last stage, shorter than BK, k clamped to kmax (last vector start).
  // records: bytes from the stage's base up to the operand's end.
  template <bool TAIL>
  __device__ __forceinline__ void issue(gptr<const T> P, uint32_t records, int64_t ld, int64_t k0, int64_t kmax, int wave,
                                        int lane, char* dst, int i) const {
    const int p = wave + NW * i;
    const int kleft = TAIL ? (int)(kmax - k0) : BK;
    const int kp = krow<TAIL>(p, kleft);
    Off o = off[i];
    if (TAIL) {
      asm volatile("" : "+v"(lane));  // the clamps are formed here, not ahead of the main loop
      o -= past(p, kp, kleft, ld, lane);
    }
    if constexpr (WIDE) {
      gptr<const char> src = (gptr<const char>)(P + (RC ? (k0 + kp) * ld : k0)) + o;
      __builtin_amdgcn_global_load_lds((gptr<const void>)src, (JB_LDS void*)(dst + p * PB), 4, 0, 0);
    } else {
      // A buffer load adds the stage's base (descriptor), the load's offset (scalar)
      // and the lane's by itself: no vector address arithmetic is left in the loop.
      gptr<const T> base = P + (RC ? k0 * ld : k0);
      ring_load(base, records, o, (uint32_t)kp * (uint32_t)ld * EB, dst + p * PB);
    }
  }
};

// s_waitcnt: at most N vector-memory operations outstanding and every LDS read returned.
template <int N>
__device__ __forceinline__ void wait_ring() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}

template <typename T, bool TA, bool TB, bool WIDE, int BTM, int BTN, int WGM, int WGN, int BK, int NSLOT_>
struct RingTile {
  static constexpr int NW = WGM * WGN;  // waves
  static constexpr int NTH = 64 * NW;
  typedef RingOperand<T, BTM, BK, !TA, NW, WIDE> OA;
  typedef RingOperand<T, BTN, BK, TB, NW, WIDE> OB;
  static constexpr int WIM = BTM / WGM / 16, WIN = BTN / WGN / 16;  // 16 x 16 MFMA blocks per wave along m, n
  static constexpr int STAGE_B = OA::BYTES + OB::BYTES;
  static constexpr int NLD = OA::NP + OB::NP;  // loads per wave and stage
  // the loads a wait leaves in flight fit its counter
  static constexpr int NSLOT = (NSLOT_ - 2) * NLD < 64 ? NSLOT_ : 63 / NLD + 2;
  static constexpr int SMEM = NSLOT * STAGE_B;
  static constexpr int VW = WIDE ? 1 : 16 / (int)sizeof(T);
  static constexpr int NT4 = BK / 4;  // MFMA k-groups per stage
  static_assert(NT4 % 2 == 0, "the fragment buffers alternate over whole stages");
  typedef typename Mfma<T>::acc_t acc_t;
  typedef acc_t Acc[WIM][WIN];

  char* ring;
  int lane, wave, wm, wn, g, l16;
  gptr<const T> At, Bt;
  uint32_t arec, brec;    // bytes from the last stage's base to the operand's end,
  uint32_t arec2, brec2;  // and from the base of the one before (RingOperand::REACH; other stages' vectors end inside it)
  int64_t lda, ldb, K, kamax, kbmax;
  int ramax, rbmax, nst, nfull;
  OA oa;
  OB ob;
  T a[2][WIM], b[2][WIN];

  // smem: SMEM bytes of LDS; tid: thread index
  __device__ __forceinline__ RingTile(char* smem, int tid) : ring(smem) {
    lane = tid % 64;
    wave = __builtin_amdgcn_readfirstlane(tid / 64);
    wm = wave % WGM;
    wn = wave / WGM;
    g = lane / 16;
    l16 = lane % 16;
  }
  // The waves' blocks interleave: this lane's tile row in block row i, tile column of item r in block column j.
  __device__ __forceinline__ int row(int i) const { return 16 * (i * WGM + wm) + l16; }
  __device__ __forceinline__ int col(int j, int r) const { return 16 * (j * WGN + wn) + Mfma<T>::prow(r, g); }

  // load i of stage st; tail: the last stage, shorter than BK
  template <typename Tail>
  __device__ __forceinline__ void issue(int st, int slot, int i, Tail) const {
    char* dst = ring + slot * STAGE_B;
    const int64_t k0 = (int64_t)st * BK;
    uint32_t records = st == nst - 1 ? (i < OA::NP ? arec : brec) : 0xffffffffu;
    if constexpr (OA::REACH || OB::REACH)
      if (st == nst - 2) records = i < OA::NP ? arec2 : brec2;
    if (i < OA::NP) oa.template issue<Tail::value>(At, records, lda, k0, kamax, wave, lane, dst, i);
    else ob.template issue<Tail::value>(Bt, records, ldb, k0, kbmax, wave, lane, dst + OA::BYTES, i - OA::NP);
  }

  // min(x, most) of a uniform x >= 0
  static __device__ __forceinline__ int at_most(int64_t x, int most) {
    return upper_half(x) != 0 ? most : (int)min((uint32_t)x, (uint32_t)most);
  }
  // Takes a product: A_, B_ at the tile's first row and column and its first k; rows, cols: what is left of C
  // from there (>= 1); K_: k steps (K_ == 0: no products).  Issues the first stages' loads: every wave of the
  // block must be done with the ring.
  __device__ __forceinline__ void begin(gptr<const T> A_, int64_t lda_, gptr<const T> B_, int64_t ldb_, int64_t rows,
                                        int64_t cols, int64_t K_) {
    At = A_;
    Bt = B_;
    lda = lda_;
    ldb = ldb_;
    K = K_;
    // the last vector starts
    ramax = at_most(rows - 1, BTM) & ~(TA ? 0 : VW - 1);
    rbmax = at_most(cols - 1, BTN) & ~(TB ? VW - 1 : 0);
    kamax = (K - 1) & ~(int64_t)(TA ? VW - 1 : 0);
    kbmax = (K - 1) & ~(int64_t)(TB ? 0 : VW - 1);
    nst = (int)((uint64_t)(K + BK - 1) / BK);
    nfull = (int)((uint64_t)K / BK);
    const int64_t kr = K - (int64_t)(nst - 1) * BK;  // k of the last stage
    arec = buffer_records<T>(OA::extent(lda, rows, kr));
    brec = buffer_records<T>(OB::extent(ldb, cols, kr));
    arec2 = OA::REACH ? buffer_records<T>(OA::extent(lda, rows, kr + BK)) : 0xffffffffu;
    brec2 = OB::REACH ? buffer_records<T>(OB::extent(ldb, cols, kr + BK)) : 0xffffffffu;
    oa.init(lda, ramax, wave, lane);
    ob.init(ldb, rbmax, wave, lane);
    // The whole stages' loads and the short one's are apart, here and in stage(): with both forms of a load in one
    // branch the compiler merged their descriptors into vector registers and looped over the values.
#pragma unroll
    for (int d = 0; d < NSLOT; ++d)
      if (d < nfull) {
#pragma unroll
        for (int i = 0; i < NLD; ++i) issue(d, d, i, std::false_type());
      }
    if (nfull < nst && nfull < NSLOT) {
#pragma unroll
      for (int i = 0; i < NLD; ++i) issue(nfull, nfull, i, std::true_type());
    }
  }

  template <int WI, int WJ>
  __device__ __forceinline__ void frags(int slot, int t, T (&x)[WIM], T (&y)[WIN]) const {
    const T* as = reinterpret_cast<const T*>(ring + slot * STAGE_B);
    const T* bs = reinterpret_cast<const T*>(ring + slot * STAGE_B + OA::BYTES);
#pragma unroll
    for (int i = 0; i < WI; ++i) x[i] = as[OA::at(row(i), 4 * t + g)];
#pragma unroll
    for (int j = 0; j < WJ; ++j) y[j] = bs[OB::at(16 * (j * WGN + wn) + l16, 4 * t + g)];
  }
  // Waits for this wave's loads of stage st (all but those of the later stages in
  // flight) and its LDS reads, then for every wave.  A plain barrier: the fence of
  // __syncthreads() would wait for all loads.
  template <typename Steady>
  __device__ __forceinline__ void arrive(int st, Steady) const {
    const int later = nst - 1 - st;
    if (Steady::value || later >= NSLOT - 2) wait_ring<(NSLOT - 2) * NLD>();
    else if (NSLOT >= 4 && later == NSLOT - 3) wait_ring<(NSLOT >= 4 ? NSLOT - 3 : 0) * NLD>();
    else wait_ring<0>();
    block_barrier();
  }
  static __device__ __forceinline__ void block_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  // Stage st in slot `slot`, whose first fragments are in a[0], b[0].  In its last
  // MFMA group the block meets once: stage st + 1 has landed and every wave has
  // read all of stage st, so its slot takes stage st + NSLOT and the next stage's
  // first fragments are read while that group's MFMAs run.
  // Tail: the short last stage.  Steady: stage st + NSLOT is a whole stage.
  template <int WI, int WJ, typename Tail, typename Steady>
  __device__ __forceinline__ void stage(Acc& acc, int st, int slot, int nslot, Tail, Steady steady) {
    constexpr bool TAIL = Tail::value, STEADY = Steady::value;
#pragma unroll
    for (int t = 0; t < NT4; ++t) {
      const int cur = t & 1;
      if (TAIL) {
        if (t > 0 && (int64_t)st * BK + 4 * t >= K) return;  // only padding is left
        const bool past = (int64_t)st * BK + 4 * t + g >= K;
#pragma unroll
        for (int i = 0; i < WI; ++i) a[cur][i] = past ? T(-0.0) : a[cur][i];
#pragma unroll
        for (int j = 0; j < WJ; ++j) b[cur][j] = past ? T(0.0) : b[cur][j];
      }
      // The next group's fragments are read behind the first row of MFMAs (whose
      // wait for this group's then covers nothing else).
      if (WI == 1) ahead<WI, WJ>(st, slot, nslot, t, steady);
      // D'[p][q] = sum_k X[p][k] Y[k][q] with X = op(B)^T block (p -> n) and Y = op(A)^T
      // block (q -> m), so a 16-lane group holds 16 consecutive rows of one column of C
      // (coalesced column-major stores).
#pragma unroll
      for (int i = 0; i < WI; ++i) {
#pragma unroll
        for (int j = 0; j < WJ; ++j) acc[i][j] = Mfma<T>::mma(b[cur][j], a[cur][i], acc[i][j]);
        __builtin_amdgcn_sched_barrier(SCHED_ALU);
        if (i == 0 && WI > 1) ahead<WI, WJ>(st, slot, nslot, t, steady);
        if (t + 1 == NT4) {
          constexpr int PI = (NLD + WI - 1) / WI;
#pragma unroll
          for (int q = PI * i; q < PI * (i + 1) && q < NLD; ++q)
            if (STEADY || (!TAIL && st + NSLOT < nfull)) issue(st + NSLOT, slot, q, std::false_type());
          if (!STEADY && !TAIL && st + NSLOT >= nfull && st + NSLOT < nst) {
#pragma unroll
            for (int q = PI * i; q < PI * (i + 1) && q < NLD; ++q) issue(st + NSLOT, slot, q, std::true_type());
          }
        }
      }
      __builtin_amdgcn_sched_barrier(SCHED_ALU);
    }
  }
  // The fragments of the group after group t of stage st.
  template <int WI, int WJ, typename Steady>
  __device__ __forceinline__ void ahead(int st, int slot, int nslot, int t, Steady steady) {
    const int nxt = (t & 1) ^ 1;
    if (t + 1 < NT4) {
      frags<WI, WJ>(slot, t + 1, a[nxt], b[nxt]);
    } else if (Steady::value || st + 1 < nst) {
      arrive(st + 1, steady);
      frags<WI, WJ>(nslot, 0, a[nxt], b[nxt]);
    }
    __builtin_amdgcn_sched_barrier(SCHED_ALU);
  }
  // acc += the product; the waves may still be reading the ring when it returns.
  // WI x WJ: the blocks of each wave that are multiplied.
  template <int WI = WIM, int WJ = WIN>
  __device__ __forceinline__ void run(Acc& acc) {
    arrive(0, std::false_type());
    frags<WI, WJ>(0, 0, a[0], b[0]);
    int st = 0;
    // unrolled over the ring, so that every LDS address is a constant offset from a few lane registers
    for (; st + 2 * NSLOT - 1 < nfull; st += NSLOT)
#pragma unroll
      for (int d = 0; d < NSLOT; ++d)
        stage<WI, WJ>(acc, st + d, d, d + 1 == NSLOT ? 0 : d + 1, std::false_type(), std::true_type());
    int slot = 0, nslot = 1;
    if constexpr (WIM * WIN == 1) {
      // the last stages on constant offsets too: all of them where K is short, and little code for this tile
      for (; st < nfull; st += NSLOT)
#pragma unroll
        for (int d = 0; d < NSLOT; ++d)
          if (st + d < nfull)
            stage<WI, WJ>(acc, st + d, d, d + 1 == NSLOT ? 0 : d + 1, std::false_type(), std::false_type());
      st = nfull;
      slot = nfull % NSLOT;
    }
    for (; st < nfull; ++st) {
      stage<WI, WJ>(acc, st, slot, nslot, std::false_type(), std::false_type());
      slot = nslot;
      nslot = nslot + 1 == NSLOT ? 0 : nslot + 1;
    }
    if (st < nst) stage<WI, WJ>(acc, st, slot, nslot, std::true_type(), std::false_type());
  }
  // C = alpha*acc + beta*C on rows x cols of C from C0 (this tile's first element).
  // Buffer stores: base in a descriptor, columns in scalar offsets, one lane offset
  // for all, so that a whole tile takes one multiply and one store per element (the
  // addresses and bounds of the pointer form cost about 15 vector instructions).
  __device__ __forceinline__ void store(const Acc& acc, T* C0, int64_t ldc, int64_t rows, int64_t cols, T alpha,
                                        T beta) const {
#ifdef __HIP_DEVICE_COMPILE__  // the descriptor type exists on the device only
    typedef typename std::conditional<sizeof(T) == 8, u2v, uint32_t>::type Bits;
    if (ldc < ((int64_t)1 << 32) / ((int64_t)sizeof(T) * BTN)) {
      __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)C0, 0, 0xffffffffu, 0x00027000);
      const uint32_t ld = (uint32_t)ldc * sizeof(T);
      const uint32_t vo = (uint32_t)row(0) * sizeof(T) + (uint32_t)Mfma<T>::prow(0, g) * ld;
      auto so = [&](int j, int r) { return (16 * (j * WGN + wn) + Mfma<T>::prow(r, 0)) * ld; };
      auto get = [&](int i, int j, int r) __attribute__((always_inline)) {
        const uint32_t v = vo + 16 * WGM * i * (uint32_t)sizeof(T);
        if constexpr (sizeof(T) == 8) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rsrc, v, so(j, r), 0));
        else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rsrc, v, so(j, r), 0));
      };
      auto put = [&](int i, int j, int r, T c) __attribute__((always_inline)) {
        const uint32_t v = vo + 16 * WGM * i * (uint32_t)sizeof(T);
        if constexpr (sizeof(T) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(Bits, c), rsrc, v, so(j, r), 0);
        else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(Bits, c), rsrc, v, so(j, r), 0);
      };
      if (rows >= BTM && cols >= BTN) {
#pragma unroll
        for (int i = 0; i < WIM; ++i) {
          T cv[WIN][4];  // the beta*C loads of a block row are in flight together
          if (beta != T(0)) {
#pragma unroll
            for (int j = 0; j < WIN; ++j)
#pragma unroll
              for (int r = 0; r < 4; ++r) cv[j][r] = get(i, j, r);
          }
#pragma unroll
          for (int j = 0; j < WIN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              T c = alpha * acc[i][j][r];
              if (beta != T(0)) c = fma(beta, cv[j][r], c);
              put(i, j, r, c);
            }
        }
      } else {
#pragma unroll
        for (int j = 0; j < WIN; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (col(j, r) < cols) {
#pragma unroll
              for (int i = 0; i < WIM; ++i)
                if (row(i) < rows) {
                  T c = alpha * acc[i][j][r];
                  if (beta != T(0)) c = fma(beta, get(i, j, r), c);
                  put(i, j, r, c);
                }
            }
      }
      return;
    }
    gptr<T> C = as_global(C0);
#pragma unroll
    for (int i = 0; i < WIM; ++i)
#pragma unroll
      for (int j = 0; j < WIN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (row(i) < rows && col(j, r) < cols) {
            gptr<T> p = C + row(i) + col(j, r) * ldc;
            T c = alpha * acc[i][j][r];
            if (beta != T(0)) c = fma(beta, *p, c);
            *p = c;
          }
#endif
  }
  // The same with as many blocks per wave as reach into `rows` x `cols` of C, in
  // steps of SI x SJ: a loop of its own for each count (a branch per block inside
  // one loop cost more than the blocks it skipped: copies of the accumulators).
  template <int SI, int SJ, int WI = WIM, int WJ = WIN>
  __device__ __forceinline__ void run_fringe(Acc& acc, int64_t rows, int64_t cols) {
    if constexpr (WI > SI) {
      if (rows <= 16 * WGM * (WI - SI)) return run_fringe<SI, SJ, WI - SI, WJ>(acc, rows, cols);
    }
    if constexpr (WJ > SJ) {
      if (cols <= 16 * WGN * (WJ - SJ)) return run_fringe<SI, SJ, WI, WJ - SJ>(acc, rows, cols);
    }
    run<WI, WJ>(acc);
  }
};

}  // namespace
}  // namespace jb
