// Tile order and the LDS-staged epilogue of the tiled GEMM kernels.
#pragma once

#include <type_traits>

#include "gemm_common.h"

namespace sph {
namespace {

template <typename T>
__device__ inline f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (sizeof(T) == 2 && __is_same(T, half_t)) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(
        __builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
}

// Maps the linear workgroup id to a (tile_m, tile_n) pair: ids are first
// regrouped so that consecutive ids run on one XCD (dispatch is round-robin
// over 8 XCDs), then walked in GROUP_M-row bands for L2 reuse.
__device__ inline void tile_of(int bid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int nt = tiles_m * tiles_n;
  if ((nt & 7) == 0) bid = (bid & 7) * (nt >> 3) + (bid >> 3);
  constexpr int GROUP_M = 4;
  const int per_group = GROUP_M * tiles_n;
  const int g = bid / per_group;
  const int first_m = g * GROUP_M;
  const int gm = (tiles_m - first_m) < GROUP_M ? (tiles_m - first_m) : GROUP_M;
  const int in_g = bid - g * per_group;
  tm = first_m + in_g % gm;
  tn = in_g / gm;
}

// Writes one 32 x WTN slab of fp32 results (LDS, row pitch EPITCH floats)
// to D rows row0.., columns col0.. as D = epi(alpha * slab + beta * C).
// Lane l handles columns 8*(l % (WTN/8)) .. +7 of rows l / (WTN/8) + k*RPP.
// The activation and the C term are resolved outside the row loop.  A
// row-major C with 16-byte aligned rows (a residual, or a bias row with
// ldc_row 0) is read 16 bytes a lane, every row of the slab before the
// first store, so the slab waits for one C load latency instead of one per
// row (2048 x 4096 x 4096 + residual in 128-wide tiles: 76 -> 64 us).
template <typename T, int EPI, bool USE_C, int WTN, int EPITCH>
__device__ __attribute__((always_inline)) inline void store_slab_impl(const GemmArgs& p, const float* slab, T* D,
                                       const T* C, int64_t row0, int64_t col0,
                                       int lane) {
  constexpr int LPR = WTN / 8;   // lanes per row
  constexpr int RPP = 64 / LPR;  // rows per pass (48-wide slabs: 10, lanes 60-63 idle)
  const int er = lane / LPR, ec = (lane % LPR) * 8;
  const int64_t col = col0 + ec;
  if (er >= RPP || col >= p.n) return;
  const bool full_cols = col + 8 <= p.n;
  const int ncols = p.n - col >= 8 ? 8 : static_cast<int>(p.n - col);
  // Lanes whose 8-column group has bit 3 set read the two 16-byte halves
  // in the opposite order, so each LDS read cycle touches 64 distinct banks.
  const int sw = (lane >> 3) & 1;
  // one row: cv holds the row's 8 C values as 16 bytes when vec_c (else C
  // is read element by element, when there is a C term)
  auto row_out = [&](int rr, int64_t row, u32x4 cv, bool vec_c) __attribute__((always_inline)) {
    const u32x4* sp = reinterpret_cast<const u32x4*>(slab + rr * EPITCH + ec);
    const u32x4 h0 = sp[sw], h1 = sp[sw ^ 1];
    float v[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = __uint_as_float(sw ? h1[e] : h0[e]);
      v[e + 4] = __uint_as_float(sw ? h0[e] : h1[e]);
    }
    float cf[8];
    if constexpr (USE_C) {
      if (vec_c) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t b16 = (cv[e >> 1] >> (16 * (e & 1))) & 0xffffu;
          if constexpr (__is_same(T, bf16_t))
            cf[e] = __uint_as_float(b16 << 16);
          else
            cf[e] = static_cast<float>(__builtin_bit_cast(half_t, static_cast<uint16_t>(b16)));
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          cf[e] = e < ncols ? Num<T>::to_f(C[row * p.ldc_row + (col + e) * p.ldc_col]) : 0.f;
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float x = p.alpha * v[e];
      if constexpr (USE_C) x += p.beta * cf[e];
      if constexpr (EPI == SPH_EPI_RELU) x = fmaxf(x, 0.f);
      if constexpr (EPI == SPH_EPI_GELU) x = gelu_erf(x);
      if constexpr (EPI == SPH_EPI_SILU) x = silu(x);
      v[e] = x;
    }
    T* dp = D + row * p.ldd + col;
    // streaming stores: a launch's tiles tend to finish together, so the
    // output leaves in one burst (4096^3: 1305-1316 -> 1335-1337 TFLOP/s,
    // alternating builds on one box; the c4 / c5 decoder unchanged)
    if (full_cols)
      p.vec_d ? store8<T, true>(dp, v) : store8u<T, true>(dp, v);
    else
      store8_partial<T>(dp, ncols, v);
  };
  if constexpr (USE_C && sizeof(T) == 2) {
    if (full_cols && p.ldc_col == 1 && (p.ldc_row & 7) == 0 &&
        (reinterpret_cast<uintptr_t>(C) & 15) == 0) {
      constexpr int NR = (32 + RPP - 1) / RPP;  // row passes per slab
      u32x4 cq[NR];
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int rr = er + i * RPP;
        if (rr < 32 && row0 + rr < p.m)
          cq[i] = *reinterpret_cast<const u32x4*>(C + (row0 + rr) * p.ldc_row + col);
      }
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int rr = er + i * RPP;
        if (rr < 32 && row0 + rr < p.m) row_out(rr, row0 + rr, cq[i], true);
      }
      return;
    }
  }
#pragma unroll 1
  for (int rr = er; rr < 32; rr += RPP) {
    const int64_t row = row0 + rr;
    if (row >= p.m) break;
    row_out(rr, row, u32x4{0, 0, 0, 0}, false);
  }
}

// Calls f(std::integral_constant<int, E>, std::bool_constant<USE_C>) for the
// call's activation E and C term, so that a kernel's epilogue loop (which
// calls store_slab_impl<T, E, USE_C, ..> per 32-row slab) is instantiated
// once per case.  With the choice made inside the loop instead, the bf16
// loop bodies grew past the unroller's limit and the accumulators, indexed
// by the slab number, were kept in scratch memory.
template <typename F>
__device__ inline void epi_dispatch(const GemmArgs& p, const void* c, F&& f) {
  const bool use_c = c != nullptr && p.beta != 0.f;
#define SPH_EPI_CASE(E)                                                            \
  if (use_c)                                                                       \
    f(std::integral_constant<int, E>{}, std::true_type{});                         \
  else                                                                             \
    f(std::integral_constant<int, E>{}, std::false_type{});
  switch (p.epilogue) {
    case SPH_EPI_RELU:
      SPH_EPI_CASE(SPH_EPI_RELU);
      break;
    case SPH_EPI_GELU:
      SPH_EPI_CASE(SPH_EPI_GELU);
      break;
    case SPH_EPI_SILU:
      SPH_EPI_CASE(SPH_EPI_SILU);
      break;
    default:
      SPH_EPI_CASE(SPH_EPI_NONE);
  }
#undef SPH_EPI_CASE
}

}  // namespace
}  // namespace sph
