// jb_internal.h -- shared declarations of the HIP kernels' host launchers and
// the runtime (not part of the public C ABI; see include/jblas_hip.h).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace jb {

// Element type and transposition of one GEMM operand.
struct GemmArgs {
  bool ta, tb;          // op(A) = A^T, op(B) = B^T
  int64_t m, n, k;
  double alpha, beta;
  const void* A;
  int64_t lda;
  const void* B;
  int64_t ldb;
  void* C;
  int64_t ldc;
  // Split-K (adjoints of small products): k per split, a multiple of 32 (0: one
  // chain over all of k), device memory for the splits' results (else null) and zeroed per-tile
  // counters (gemm_mfma_split_need / bf16x3_split_need), which the call leaves zeroed.
  int64_t kchunk = 0;
  void* part = nullptr;
  int* counters = nullptr;
};
int gemm_splits(const GemmArgs& g);

// ---- FP64 -----------------------------------------------------------------
// Native FP64 MFMA GEMM; its chains are the jmul! recurrence bit for bit.
hipError_t launch_dgemm_mfma(const GemmArgs& g, hipStream_t s);
// The jmul! recurrence on the vector ALUs (sequential fma).
hipError_t launch_dgemm_recurrence(const GemmArgs& g, hipStream_t s);
// kernel! (D += A*X) on the FP64 MFMA kernel: each chain starts from C and
// every step is an fma; alpha/beta unused.
hipError_t launch_dgemm_mfma_acc(const GemmArgs& g, hipStream_t s);
// C = beta*C (alpha == 0 or k == 0 quick path); beta == 0 writes zeros.
hipError_t launch_scale_f64(int64_t m, int64_t n, double beta, double* C, int64_t ldc, hipStream_t s);
hipError_t launch_scale_f32(int64_t m, int64_t n, float beta, float* C, int64_t ldc, hipStream_t s);
// Whole-matrix small GEMM D = A*X (fastmul!), one fma chain per element.
hipError_t launch_fastmul_f64(int64_t M, int64_t N, int64_t P, double* D, const double* A, const double* X,
                              hipStream_t s);
hipError_t launch_fastmul_f32(int64_t M, int64_t N, int64_t P, float* D, const float* A, const float* X,
                              hipStream_t s);

// ---- split-BF16 emulated FP64 --------------------------------------------
// Workspace bytes needed for an m x n x k problem with s slices.
size_t ozaki_workspace_bytes(int64_t m, int64_t n, int64_t k, int s);
// Split + slice-pair GEMM + compensated combine.  `ws` is device memory of
// ozaki_workspace_bytes().  A row of op(A) or column of op(B) holding Inf or
// NaN makes the C elements it feeds NaN and sets two device ints to 1: with
// `want_flag` this call's, an int at byte offset emulated_flag_offset() of `ws` (cleared
// by the call itself), and `sticky`, which the call never clears.  No host
// synchronisation.
hipError_t launch_dgemm_ozaki(const GemmArgs& g, int s, void* ws, bool want_flag, int* sticky, hipStream_t st);
// The same with INT8 slices (v_mfma_i32_32x32x32_i8, exact int32 level sums).
size_t ozaki_i8_workspace_bytes(int64_t m, int64_t n, int64_t k, int s);
hipError_t launch_dgemm_ozaki_i8(const GemmArgs& g, int s, void* ws, bool want_flag, int* sticky, hipStream_t st);
// Byte offset of the call's non-finite flag in the workspace of the emulated
// DGEMM (BF16 or INT8 slices) and of the 3xBF16 SGEMM (whose planes have their
// own layout).
size_t emulated_flag_offset(int64_t m, int64_t n, int64_t k, int s, bool i8);
size_t bf16x3_flag_offset(int64_t m, int64_t n, int64_t k);

// ---- FP32 -----------------------------------------------------------------
// Native FP32 MFMA GEMM; its chains are the jmul! recurrence in Float32 bit for bit.
hipError_t launch_sgemm_mfma(const GemmArgs& g, hipStream_t s);
// Device memory a split-K product on launch_dgemm_mfma (elt 8) / launch_sgemm_mfma (elt 4) needs.
void gemm_mfma_split_need(const GemmArgs& g, size_t elt, size_t* part_bytes, int64_t* counters);
void bf16x3_split_need(const GemmArgs& g, size_t* part_bytes, int64_t* counters);
size_t bf16x3_workspace_bytes(int64_t m, int64_t n, int64_t k, int splits = 1);
// Non-finite inputs become NaN slices (every product they enter is NaN) and set
// the two flags as in launch_dgemm_ozaki.
hipError_t launch_sgemm_bf16x3(const GemmArgs& g, int nprod, void* ws, bool want_flag, int* sticky, hipStream_t s);

// p[0..n) = 0, n >= 1: a kernel, since a captured graph takes no memset.
hipError_t launch_zero_i32(int* p, int64_t n, hipStream_t s);

// ---- generator ------------------------------------------------------------
hipError_t launch_fill_uniform(uint64_t seed, int64_t n, double* out, hipStream_t s);
hipError_t launch_fill_uniform_f32(uint64_t seed, int64_t n, float* out, hipStream_t s);
hipError_t launch_fill_wide(uint64_t seed, int64_t n, int emin, int emax, double* out, hipStream_t s);
hipError_t launch_fill_wide_f32(uint64_t seed, int64_t n, int emin, int emax, float* out, hipStream_t s);
hipError_t launch_fill_normal(uint64_t seed, int64_t n, double scale, double* out, hipStream_t s);
hipError_t launch_fill_normal_f32(uint64_t seed, int64_t n, double scale, float* out, hipStream_t s);

// Compute units of the runtime's device (from the device query at init);
// launch geometry that depends on the device reads it.
int runtime_compute_units();

// Per-kernel timing (off unless jb_kernel_timing_enable(1)): HIP events
// recorded on the launch stream around one kernel launch.  Not recorded while
// the stream is being captured into a graph.
void timing_begin(hipStream_t s, const char* kernel);
void timing_end(hipStream_t s, const char* kernel);

// Pointers that a kernel reads from memory (a descriptor, a struct argument)
// carry no address space the compiler can infer, so accesses through them are
// flat accesses, which also count against the LDS wait counter (a wait for an
// LDS read then waits for outstanding global traffic too).  Casting them to
// the global address space gives global loads and stores.
template <typename T> using gptr = __attribute__((address_space(1))) T*;
template <typename T> __device__ __forceinline__ gptr<T> as_global(T* p) { return (gptr<T>)p; }

// Upper half of a uniform x, kept apart from it: comparisons of it are scalar instructions,
// those of 64-bit numbers vector ones.
__device__ __forceinline__ int upper_half(int64_t x) {
  int hi = __builtin_amdgcn_readfirstlane((int)(x >> 32));
  asm("" : "+s"(hi));
  return hi;
}

// Record count of a buffer descriptor over `elements` of T, at most 2^32 - 1.
template <typename T> __device__ __forceinline__ uint32_t buffer_records(int64_t elements) {
  const int64_t bytes = elements * (int64_t)sizeof(T);
  return (uint32_t)__builtin_amdgcn_readfirstlane(upper_half(bytes) != 0 ? -1 : (int)bytes);
}

// Split-K partial results pass between workgroups on different XCDs, whose L2s are not
// coherent.  Device-scope stores and loads of the elements themselves (write-through,
// read past the L2), the stores drained before the tile's arrival counter is raised,
// take the place of device-scope fences: a fence writes the whole L2 back, and every
// wave of every split issued one (256 x 384 x 512 FP32 in two splits: 25.9 us, 8.1 so;
// 1024 uneven FP64 products of a plan 2405, 2380).
template <typename T> __device__ __forceinline__ void agent_store(gptr<T> p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> __device__ __forceinline__ T agent_load(gptr<const T> p) {
  return __hip_atomic_load((gptr<T>)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void drain_stores() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// XCD-aware block swizzle: hardware places workgroup w on XCD (w % nxcd).
// Returns a tile id such that each XCD owns a contiguous range of tile ids.
__device__ __forceinline__ int xcd_remap(int w, int nblocks, int nxcd) {
  const int q = nblocks / nxcd, r = nblocks % nxcd;
  const int x = w % nxcd, local = w / nxcd;
  return (x < r) ? x * (q + 1) + local : r * (q + 1) + (x - r) * q + local;
}

// Grouped ordering of an (tm x tn) tile grid: GROUP tile-rows walked column by
// column so that concurrently running tiles share A row panels and B column panels.
__device__ __forceinline__ void tile_coords(int tile, int tiles_m, int tiles_n, int group, int& tm, int& tn) {
  const int per_group = group * tiles_n;
  const int gid = tile / per_group;
  const int first_m = gid * group;
  const int gsize = min(tiles_m - first_m, group);
  const int in_group = tile - gid * per_group;
  tm = first_m + in_group % gsize;
  tn = in_group / gsize;
}

}  // namespace jb
