// What the GEMM translation units share: the call's arguments, the MFMA and
// LDS-DMA primitives and the scalar epilogue.
#pragma once

#include "sph_common.h"

namespace sph {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct GemmArgs {
  int64_t m, n, k;
  const void* a;
  int64_t lda, stride_a;
  const void* b;
  int64_t ldb, stride_b;
  const void* c;
  int64_t ldc_row, ldc_col, stride_c;
  void* d;
  int64_t ldd, stride_d;
  float alpha, beta;
  int epilogue;
  int vec_a, vec_b, vec_d;
  int tiles_m, tiles_n;
  // Split-K tail (direct-load kernel): tiles ranked tail_start.. run as
  // `splits` workgroups each, over kslice K tiles apiece, writing fp32
  // partial tiles to part[(rank - tail_start) * splits + split] that
  // gemm_splitk_reduce sums.  tail_start = the tile count: no split.
  int tail_start, splits, kslice;
  float* part;
  int64_t part_bytes;
  // RMSNorm prologue of the small-M kernels (decode): with norm_w set, row m
  // of A enters the product as A[m] * norm_w * rsqrt(mean(A[m]^2) + norm_eps).
  // The weight multiplies each A chunk as it is loaded (rounded to the
  // element type, as a separate norm kernel's output would be); the row scale
  // multiplies the finished sums, its sum of squares accumulated alongside
  // them from the same loads.
  const void* norm_w;
  float norm_eps;
  // Batch entries (persistent kernels, whose grid does not carry them).
  int64_t batches;
  // Readable columns of a row-major B's rows (n, or n padded to whole chunks).
  int64_t nb;
};

namespace {

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
#define SPH_LDS __attribute__((address_space(3)))

// Raw buffer resource over [base, base + bytes) (stride 0; gfx9 dword 3).
__device__ inline i32x4 buffer_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  i32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(static_cast<uint32_t>(a)));
  r[1] = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(static_cast<uint32_t>(a >> 32) & 0xffffu));
  r[2] = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(bytes));
  r[3] = 0x00020000;
  return r;
}

// 16 bytes per lane from rsrc[voff + soff] into LDS at lds_addr + 16 * lane.
__device__ inline void dma16(i32x4 rsrc, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(lds_addr), "v"(voff), "s"(rsrc), "s"(soff)
               : "memory", "m0");
}
template <int N>
__device__ inline void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ inline void wait_lgkmcnt0() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

__device__ inline u32x4 zero4() {
  u32x4 z = {0u, 0u, 0u, 0u};
  return z;
}

template <typename T>
__device__ inline f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (__is_same(T, half_t)) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(
        __builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
}


// Row-major B: K row k's 16-byte chunk c sits at slot c ^ bswz(k).  A
// transposing read's 32-lane half covers rows k0 .. k0 + 3 and k0 + 8 ..
// k0 + 11 (k0 a multiple of 4 with bit 3 clear) at the same two chunks:
// bits 2-3 of the XOR spread the four rows of a lane group over the 256
// bytes of banks, bit 1 moves the second group's rows to the other half.
__device__ inline int bswz(int k) { return 4 * (k & 3) + 2 * ((k >> 3) & 1); }

// alpha, beta * C and the activation for one output element.
template <typename T>
__device__ inline float epilogue_one(const GemmArgs& p, float v, int64_t bz, int m, int64_t n) {
  v *= p.alpha;
  if (p.c != nullptr && p.beta != 0.f) {
    const T* C = static_cast<const T*>(p.c) + bz * p.stride_c;
    v += p.beta * Num<T>::to_f(C[m * p.ldc_row + n * p.ldc_col]);
  }
  if (p.epilogue == SPH_EPI_RELU) v = fmaxf(v, 0.f);
  else if (p.epilogue == SPH_EPI_GELU) v = gelu_erf(v);
  else if (p.epilogue == SPH_EPI_SILU) v = silu(v);
  return v;
}

}  // namespace
}  // namespace sph
