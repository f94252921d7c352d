// Register-staged GEMM: any layout, size and alignment of the operands
// (v_mfma_f32_32x32x16).
//
//
// Structure
//   * Workgroup tile BM x BN, K step 64, WM x WN waves; each wave owns a
//     (BM/WM) x (BN/WN) block of 32x32 MFMA tiles whose fp32 accumulators
//     stay in registers for the whole K loop.  Whole 256x256 tiles use 8
//     waves (two per SIMD, so latency hides across waves).
//   * Both operands are staged in LDS "K-contiguous": tile row r (an M row of
//     A or an N column of B) holds its 64 K values as eight 16-byte chunks,
//     chunk c stored at slot c ^ ((r >> 1) & 7), which makes the 16-byte
//     fragment reads and the loaders' 16-byte writes free of bank conflicts
//     on gfx950's 64-bank LDS.
//   * An operand whose K is contiguous in memory (A row-major; B given as
//     B^T row-major, the nn.Linear weight layout) is copied chunk by chunk.
//     An operand whose K is strided (B row-major, A transposed) is loaded as
//     8x8 blocks (eight 16-byte rows) and transposed in registers with byte
//     permutes before the LDS write.
//   * Whole tiles (FULL) run a three-deep pipeline without bounds checks:
//     K tile k is multiplied from one LDS buffer while tile k+1 moves from
//     registers to the other buffer and tile k+2 is loaded from memory.
//     Partial tiles use bounds-checked loaders and a two-deep pipeline.
//   * The epilogue stages each 32-row slab of results in LDS and writes D
//     as whole rows with 16-byte stores; activation and the C term are
//     resolved once per slab, not per element.
//   * Workgroup ids are remapped so that the 8 XCDs (round-robin dispatch)
//     each get a compact group of C tiles, sharing A rows and B columns in
//     their own L2.
#include "gemm_route.h"
#include "gemm_tile.h"

namespace sph {
namespace {

constexpr int BK = 64;  // K per LDS stage (eight 16-byte chunks of fp16)

// Reads `n` (< 8) two-byte elements with element stride `es` into a chunk,
// zero-filling the rest.
__device__ inline u32x4 load_partial(const uint16_t* p, int n, int64_t es) {
  uint16_t e[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) e[i] = (i < n) ? p[i * es] : static_cast<uint16_t>(0);
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    r[i] = static_cast<uint32_t>(e[2 * i]) | (static_cast<uint32_t>(e[2 * i + 1]) << 16);
  return r;
}

// LDS offset (in 2-byte elements) of chunk c of tile row r.  gfx950's LDS
// serves 16 lanes of a 16-byte access per cycle from 64 four-byte banks
// (a 256-byte window): a 128-byte tile row covers one half of the window
// (even rows the low half, odd rows the high half), so the eight rows of
// each parity among 16 consecutive rows must use eight different 16-byte
// slots, which c ^ ((r >> 1) & 7) guarantees for every fixed c.
__device__ inline int lds_off(int r, int c) { return r * BK + ((c ^ ((r >> 1) & 7)) << 3); }

// ---------------------------------------------------------------------------
// Tile loaders: global -> registers (issue) and registers -> LDS (commit).
// `rows` is the tile height (BM for A, BN for B); r0 the first global row
// (M index for A, N index for B); nrows the matrix extent in that dim.
// ---------------------------------------------------------------------------

// K-contiguous operand: element (r, k) at base[r * ld + k].
template <int ROWS, int NT>
struct KContLoader {
  static constexpr int PER_T = (ROWS * 8 + NT - 1) / NT;
  static constexpr int NLOADS = PER_T;  // global loads per issue
  u32x4 reg[PER_T];

  // FULL: the whole tile is in bounds and 16-byte aligned (no checks).
  template <bool FULL>
  __device__ inline void issue(const uint16_t* __restrict__ base, int64_t ld,
                               int64_t r0, int64_t nrows, int64_t k0,
                               int64_t kdim) {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < PER_T; ++i) {
      const int idx = t + i * NT;
      const int r = idx >> 3, c = idx & 7;
      const int64_t gr = r0 + r, gk = k0 + c * 8;
      if ((ROWS * 8) % NT != 0 && idx >= ROWS * 8) continue;
      if (FULL) {
        reg[i] = *reinterpret_cast<const u32x4*>(base + gr * ld + gk);
      } else if (gr < nrows && gk + 8 <= kdim) {
        reg[i] = *reinterpret_cast<const u32x4_any*>(base + gr * ld + gk);
      } else if (gr < nrows && gk < kdim) {
        const int64_t n = kdim - gk;
        reg[i] = load_partial(base + gr * ld + gk, n > 8 ? 8 : static_cast<int>(n), 1);
      } else {
        reg[i] = zero4();
      }
    }
  }

  __device__ inline void commit(uint16_t* __restrict__ lds) const {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < PER_T; ++i) {
      const int idx = t + i * NT;
      if ((ROWS * 8) % NT != 0 && idx >= ROWS * 8) continue;
      const int r = idx >> 3, c = idx & 7;
      *reinterpret_cast<u32x4*>(lds + lds_off(r, c)) = reg[i];
    }
  }
};

// K-strided operand: element (r, k) at base[k * ld + r].  Loaded as 8x8
// blocks: block (rb, kb) covers rows 8rb..8rb+7 and k 8kb..8kb+7; the 8
// global loads are along r (16 bytes each), the block is transposed in
// registers so each LDS write is one 16-byte K chunk of one row.
template <int ROWS, int NT>
struct KStridedLoader {
  static constexpr int NB = ROWS;  // (ROWS / 8) r-blocks x 8 k-blocks
  static constexpr int PER_T = (NB + NT - 1) / NT;
  static constexpr int NLOADS = PER_T * 8;
  u32x4 reg[PER_T][8];

  template <bool FULL>
  __device__ inline void issue(const uint16_t* __restrict__ base, int64_t ld,
                               int64_t r0, int64_t nrows, int64_t k0,
                               int64_t kdim) {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < PER_T; ++i) {
      const int idx = t + i * NT;
      if (NB % NT != 0 && idx >= NB) continue;
      const int kb = idx & 7, rb = idx >> 3;
      const int64_t gr = r0 + rb * 8;
#pragma unroll
      for (int kr = 0; kr < 8; ++kr) {
        const int64_t gk = k0 + kb * 8 + kr;
        if (FULL) {
          reg[i][kr] = *reinterpret_cast<const u32x4*>(base + gk * ld + gr);
        } else if (gk < kdim && gr + 8 <= nrows) {
          reg[i][kr] = *reinterpret_cast<const u32x4_any*>(base + gk * ld + gr);
        } else if (gk < kdim && gr < nrows) {
          const int64_t n = nrows - gr;
          reg[i][kr] = load_partial(base + gk * ld + gr, n > 8 ? 8 : static_cast<int>(n), 1);
        } else {
          reg[i][kr] = zero4();
        }
      }
    }
  }

  __device__ inline void commit(uint16_t* __restrict__ lds) const {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < PER_T; ++i) {
      const int idx = t + i * NT;
      if (NB % NT != 0 && idx >= NB) continue;
      const int kb = idx & 7, rb = idx >> 3;
      // reg[i][kr] dword q holds rows (2q, 2q+1) of k row kr.  Output row j
      // (= r offset) dword p holds k values (2p, 2p+1).  Lanes of odd r
      // blocks write rows in the order 1,0,3,2,... so that the 16 lanes of
      // one LDS write cycle (two r blocks) cover rows of both parities.
      const int flip = rb & 1;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int jj = j ^ flip;
        const uint32_t sel = (jj & 1) ? 0x07060302u : 0x05040100u;
        u32x4 o;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const uint32_t lo = reg[i][2 * p][j >> 1];
          const uint32_t hi = reg[i][2 * p + 1][j >> 1];
          o[p] = __builtin_amdgcn_perm(hi, lo, sel);
        }
        const int r = rb * 8 + jj;
        *reinterpret_cast<u32x4*>(lds + lds_off(r, kb)) = o;
      }
    }
  }
};

template <bool KCONT, int ROWS, int NT>
struct LoaderSel;
template <int ROWS, int NT>
struct LoaderSel<true, ROWS, NT> {
  using type = KContLoader<ROWS, NT>;
};
template <int ROWS, int NT>
struct LoaderSel<false, ROWS, NT> {
  using type = KStridedLoader<ROWS, NT>;
};


// Reads the MFMA fragments of K sub-step kk (16 K values) for this wave.
template <int TM, int TN, int WTM, int WTN>
__device__ inline void load_frags(const uint16_t* __restrict__ sa,
                                  const uint16_t* __restrict__ sb, int wm,
                                  int wn, int row_in, int khalf, int kk,
                                  u32x4 (&af)[TM], u32x4 (&bf)[TN]) {
  const int c = kk * 2 + khalf;
#pragma unroll
  for (int i = 0; i < TM; ++i)
    af[i] = *reinterpret_cast<const u32x4*>(sa + lds_off(wm * WTM + i * 32 + row_in, c));
#pragma unroll
  for (int j = 0; j < TN; ++j)
    bf[j] = *reinterpret_cast<const u32x4*>(sb + lds_off(wn * WTN + j * 32 + row_in, c));
}

template <typename T, int BM, int BN, int WM, int WN, bool A_KCONT, bool B_KCONT,
          bool FULL>
__global__ void __launch_bounds__(WM * WN * 64)
gemm_kernel(const GemmArgs p) {
  constexpr int NT = WM * WN * 64;
  constexpr int WTM = BM / WM, WTN = BN / WN;  // wave tile
  constexpr int TM = WTM / 32;                 // 32x32 MFMA tiles per wave along M
  constexpr int TN = WTN / 32;
  constexpr int STAGE = (BM + BN) * BK;        // LDS elements per pipeline stage
  // Epilogue staging: per wave one 32-row slab of fp32 accumulators, rows
  // padded by 8 floats so the two half-waves' rows land on different banks.
  constexpr int EPITCH = WTN + 8;
  static_assert(TM >= 1 && TN >= 1, "wave tile too small");
  static_assert(WM * WN * 32 * EPITCH * 4 <= 2 * STAGE * 2, "epilogue staging exceeds LDS");
  __shared__ __attribute__((aligned(16))) uint16_t lds[2 * STAGE];

  int tm, tn;
  tile_of(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
  const int64_t batch = blockIdx.y;
  const uint16_t* A = static_cast<const uint16_t*>(p.a) + batch * p.stride_a;
  const uint16_t* B = static_cast<const uint16_t*>(p.b) + batch * p.stride_b;
  const int64_t m0 = static_cast<int64_t>(tm) * BM;
  const int64_t n0 = static_cast<int64_t>(tn) * BN;

  typename LoaderSel<A_KCONT, BM, NT>::type la;
  typename LoaderSel<B_KCONT, BN, NT>::type lb;

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int row_in = lane & 31;  // fragment row within a 32x32 tile
  const int khalf = lane >> 5;   // which 8-wide K half of a 16-K step

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int64_t ksteps = (p.k + BK - 1) / BK;
  if constexpr (FULL) {
    // Three-deep pipeline over K tiles: while the MFMAs consume tile ks
    // from LDS buffer ks&1, tile ks+1 (loaded into registers during the
    // previous step) is written to the other buffer, and tile ks+2 is
    // loaded from global memory into the freed registers.  Global loads
    // thus have a whole K step to land and the LDS writes never wait.
    // The body is branch-free (one scheduling region): indices past the
    // last tile are clamped, re-loading and re-writing the last tile into
    // the idle buffer, which nothing reads afterwards.
    const int64_t klast = (ksteps - 1) * BK;
    la.template issue<true>(A, p.lda, m0, p.m, 0, p.k);
    lb.template issue<true>(B, p.ldb, n0, p.n, 0, p.k);
    la.commit(lds);
    lb.commit(lds + BM * BK);
    const int64_t k1 = BK < klast ? BK : klast;
    la.template issue<true>(A, p.lda, m0, p.m, k1, p.k);
    lb.template issue<true>(B, p.ldb, n0, p.n, k1, p.k);
    __syncthreads();
    for (int64_t ks = 0; ks < ksteps; ++ks) {
      const int cur = static_cast<int>(ks & 1);
      const uint16_t* sa = lds + cur * STAGE;
      const uint16_t* sb = sa + BM * BK;
      u32x4 af[2][TM], bf[2][TN];
      load_frags<TM, TN, WTM, WTN>(sa, sb, wm, wn, row_in, khalf, 0, af[0], bf[0]);
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk) {
        if (kk + 1 < BK / 16)
          load_frags<TM, TN, WTM, WTN>(sa, sb, wm, wn, row_in, khalf, kk + 1,
                                       af[(kk + 1) & 1], bf[(kk + 1) & 1]);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = mfma32<T>(af[kk & 1][i], bf[kk & 1][j], acc[i][j]);
      }
      la.commit(lds + (cur ^ 1) * STAGE);
      lb.commit(lds + (cur ^ 1) * STAGE + BM * BK);
      const int64_t k2 = (ks + 2) * BK < klast ? (ks + 2) * BK : klast;
      la.template issue<true>(A, p.lda, m0, p.m, k2, p.k);
      lb.template issue<true>(B, p.ldb, n0, p.n, k2, p.k);
      // Instruction order for the scheduler (one wave per SIMD, so latency
      // must be hidden inside the wave): fragment reads of sub-step 0;
      // sub-steps 0-2 alternate MFMAs with the next sub-step's fragment
      // reads; sub-step 3 interleaves each MFMA with the register
      // transposes, LDS writes and global loads of the pipeline.
      constexpr int NMF = TM * TN, NDS = TM + TN;
      constexpr int NVM = decltype(la)::NLOADS + decltype(lb)::NLOADS;
      constexpr int IO_PER = (NVM + NMF - 1) / NMF;  // one LDS write per global load
      // Sub-step kk's MFMAs run only after all fragment reads of sub-step
      // kk+1 were issued, so those reads overlap a whole sub-step of MFMAs.
      // (With two or more waves per SIMD the hardware interleaves waves and
      // the compiler's own order is kept.)
      if constexpr (WM * WN == 4) {
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * NDS, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, NMF, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, NDS, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, NMF, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, NDS, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, NMF, 0);
#pragma unroll
      for (int x = 0; x < NMF; ++x) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        __builtin_amdgcn_sched_group_barrier(0x200, IO_PER, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, IO_PER, 0);
      }
      }
      __syncthreads();
    }
  } else {
    if (ksteps > 0) {
      la.template issue<false>(A, p.lda, m0, p.m, 0, p.k);
      lb.template issue<false>(B, p.ldb, n0, p.n, 0, p.k);
      la.commit(lds);
      lb.commit(lds + BM * BK);
      __syncthreads();
    }
    for (int64_t ks = 0; ks < ksteps; ++ks) {
      const int cur = static_cast<int>(ks & 1);
      const bool more = ks + 1 < ksteps;
      if (more) {
        la.template issue<false>(A, p.lda, m0, p.m, (ks + 1) * BK, p.k);
        lb.template issue<false>(B, p.ldb, n0, p.n, (ks + 1) * BK, p.k);
      }
      const uint16_t* sa = lds + cur * STAGE;
      const uint16_t* sb = sa + BM * BK;
      u32x4 af[2][TM], bf[2][TN];
      load_frags<TM, TN, WTM, WTN>(sa, sb, wm, wn, row_in, khalf, 0, af[0], bf[0]);
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk) {
        if (kk + 1 < BK / 16)
          load_frags<TM, TN, WTM, WTN>(sa, sb, wm, wn, row_in, khalf, kk + 1,
                                       af[(kk + 1) & 1], bf[(kk + 1) & 1]);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = mfma32<T>(af[kk & 1][i], bf[kk & 1][j], acc[i][j]);
      }
      if (more) {
        la.commit(lds + (cur ^ 1) * STAGE);
        lb.commit(lds + (cur ^ 1) * STAGE + BM * BK);
      }
      __syncthreads();
    }
  }

  // Epilogue.  Accumulator register r of tile (i, j) holds row
  // 8*(r/4) + 4*(lane/32) + r%4, column lane%32 of that 32x32 tile.  Each
  // 32-row slab of the wave tile goes through LDS so that the output is
  // written as whole rows with 16-byte stores.
  T* D = static_cast<T*>(p.d) + batch * p.stride_d;
  const T* C = p.c ? static_cast<const T*>(p.c) + batch * p.stride_c : nullptr;
  float* slab = reinterpret_cast<float*>(lds) + wave * (32 * EPITCH);
  const int64_t row0 = m0 + wm * WTM;
  const int64_t colw = n0 + wn * WTN;
  epi_dispatch(p, C, [&](auto epi_, auto use_c_) {
    constexpr int E = decltype(epi_)::value;
    constexpr bool UC = decltype(use_c_)::value;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          slab[((r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) * EPITCH + j * 32 + (lane & 31)] =
              acc[i][j][r];
      __syncthreads();
      store_slab_impl<T, E, UC, WTN, EPITCH>(p, slab, D, C, row0 + i * 32, colw, lane);
      __syncthreads();
    }
  });
}

template <typename T, int BM, int BN, int WM, int WN, bool FULL>
void launch_full(const GemmArgs& p, dim3 grid, dim3 block, bool a_kcont, bool b_kcont,
                 hipStream_t st) {
  if (a_kcont && b_kcont)
    gemm_kernel<T, BM, BN, WM, WN, true, true, FULL><<<grid, block, 0, st>>>(p);
  else if (a_kcont && !b_kcont)
    gemm_kernel<T, BM, BN, WM, WN, true, false, FULL><<<grid, block, 0, st>>>(p);
  else if (!a_kcont && b_kcont)
    gemm_kernel<T, BM, BN, WM, WN, false, true, FULL><<<grid, block, 0, st>>>(p);
  else
    gemm_kernel<T, BM, BN, WM, WN, false, false, FULL><<<grid, block, 0, st>>>(p);
}

// Launches BM x BN tiles on the register-staged kernel: whole tiles with the
// FULL variant on WMF x WNF waves, otherwise the checked one on WMP x WNP.
template <typename T, int BM, int BN, int WMF, int WNF, int WMP, int WNP>
int launch_cfg(GemmArgs& p, int64_t batch, bool a_kcont, bool b_kcont,
               hipStream_t st) {
  p.tiles_m = static_cast<int>(ceil_div(p.m, BM));
  p.tiles_n = static_cast<int>(ceil_div(p.n, BN));
  dim3 grid(static_cast<unsigned>(p.tiles_m) * p.tiles_n, static_cast<unsigned>(batch));
  // Every tile whole and every operand row 16-byte aligned: no bounds or
  // alignment checks in the K loop.
  const bool full = p.m % BM == 0 && p.n % BN == 0 && p.k % BK == 0 && p.k > 0 &&
                    p.vec_a && p.vec_b;
  if (full)
    launch_full<T, BM, BN, WMF, WNF, true>(p, grid, dim3(WMF * WNF * 64), a_kcont, b_kcont, st);
  else
    launch_full<T, BM, BN, WMP, WNP, false>(p, grid, dim3(WMP * WNP * 64), a_kcont, b_kcont, st);
  return check_launch("sph_gemm");
}

template <typename T>
int staged_t(GemmArgs& p, int64_t batch, bool a_kcont, bool b_kcont, hipStream_t st) {
  const int64_t t256 = ceil_div(p.m, 256) * ceil_div(p.n, 256) * batch;
  const int64_t t128 = ceil_div(p.m, 128) * ceil_div(p.n, 128) * batch;
  // 256x256 whole tiles run 8 waves (128x64 each, two per SIMD, so one
  // wave's LDS and global-load latency hides under the other's MFMAs);
  // partial tiles keep 4 waves, whose bounds-checked loaders need the
  // larger per-wave register budget.
  if (t256 >= 256) return launch_cfg<T, 256, 256, 2, 4, 2, 2>(p, batch, a_kcont, b_kcont, st);
  if (t128 >= 128) return launch_cfg<T, 128, 128, 2, 2, 2, 2>(p, batch, a_kcont, b_kcont, st);
  return launch_cfg<T, 64, 64, 2, 2, 2, 2>(p, batch, a_kcont, b_kcont, st);
}

}  // namespace

int launch_staged(bool bf16, GemmArgs& p, int64_t batch, bool a_kcont, bool b_kcont,
                  hipStream_t st) {
  if (bf16) return staged_t<bf16_t>(p, batch, a_kcont, b_kcont, st);
  return staged_t<half_t>(p, batch, a_kcont, b_kcont, st);
}

}  // namespace sph
