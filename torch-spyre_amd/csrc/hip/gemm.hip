// fp16 / bf16 GEMM on gfx950 MFMA, fp32 accumulate, with an alpha/beta/bias/
// activation epilogue: the choice of kernel for a call, the direct-load kernel
// of whole and ragged 256-row tiles (v_mfma_f32_16x16x32), the short-K kernels
// (v_mfma_f32_32x32x16) and the C entry points.  gemm_ring.hip holds the
// kernel of small and ragged row counts, gemm_small.hip the streaming kernels
// of few rows, gemm_staged.hip the register-staged kernel that takes
// every layout and alignment.
#include <algorithm>
#include <type_traits>

#include "gemm_route.h"
#include "gemm_tile.h"

namespace sph {
namespace {

// ---------------------------------------------------------------------------
// Whole 256-row tiles (256, 192 or 128 columns) with A K-contiguous: direct
// global -> LDS loads.
//
//   * Each 64-deep K tile moves from memory into LDS with
//     buffer_load_dwordx4 ... lds: no VGPR staging and no LDS write
//     instructions.  Lane l's 16 bytes land at line base + 16 l (one 1 KB
//     line per instruction), so the swizzled LDS layout is produced by
//     choosing which 16 global bytes each lane fetches.  The loads are
//     raw-buffer loads whose range ends where the tile's operand rows end:
//     an offset past it reads zeros instead of touching other memory.
//   * A (and a K-contiguous B) sits K-contiguous in LDS with the swizzle of
//     the register-staged kernel.  A row-major B ([K, N], N contiguous) sits
//     as 64 K rows of 256 N values; its MFMA fragments are read with
//     ds_read_b64_tr_b16, which works on groups of 16 lanes: lane 4e + q
//     points at 4 consecutive values of one row and lane i receives value
//     i % 4 of the rows addressed by lanes i / 4, 4 + i / 4, 8 + i / 4,
//     12 + i / 4.  Pointing lane 4e + q at (k0 + e, n0 + 4q) therefore gives
//     lane i the column n0 + i at k0 .. k0 + 3, half of a B fragment.  Row
//     k's 16-byte chunk c is stored at slot c ^ bswz(k) (4 (k & 3) + 2
//     (bit 3 of k)): the 8 rows x 2 chunks a half-wave reads then cover all
//     64 banks.  (With c ^ 4 (k & 3) alone, rows k and k + 8 share banks:
//     27 % of the LDS-active cycles were bank conflicts.)
//   * 16x16x32 MFMAs (v_mfma_f32_16x16x32_{f16,bf16}), not 32x32x16: the
//     same FLOPs per LDS byte for a given wave tile, but a quarter of the
//     accumulator registers per instruction.  This part runs the GEMM at
//     its power limit, and a loop of nothing but MFMAs sustains 2006
//     TFLOP/s with 16x16x32 against 1705 with 32x32x16 (8 waves per CU,
//     random operands); the kernel gained 5-10 % on every measured shape.
//   * Two LDS stages.  The K step is ordered by hand (sched_barrier): each of
//     the two 32-deep MFMA sub-steps issues its 32 MFMAs interleaved with
//     the LDS reads of the next sub-step's fragments (B first, each A tile
//     right after this sub-step's last use of the same A index).  Early in
//     sub-step 1 a wave waits for its own DMA of the next tile and its own
//     LDS reads, then joins the barrier; the rest of sub-step 1 issues the
//     DMA of the tile after next into the stage just vacated (one line
//     every two or three MFMAs: ~1 % faster than back to back) and reads
//     the next tile's first fragments.  Past the last tile the DMA re-loads the
//     last tile and the fragment reads fetch values nobody uses, so the
//     loop has no branches.
//   * The DMA is issued from inline asm: as an intrinsic, the compiler waits
//     for every outstanding LDS DMA before any later LDS read (it cannot tell
//     the stages apart), which would serialise load and compute.  Completion
//     is awaited explicitly (vmcnt) before the barrier.
//   * 8 waves (2 x 4, two per SIMD), each owning a 128 x 64 block of 16x16
//     MFMA tiles (128 x 48 on 192-wide tiles, 128 x 32 on 128-wide ones);
//     epilogue as in the register-staged kernel.
// ---------------------------------------------------------------------------
namespace dl {
// Shared by both tile widths: 256-row tiles, 64-deep K tiles, two waves
// along M, each wave owning a 128 x 64 block of 16x16 MFMA tiles
// (v_mfma_f32_16x16x32: two 32-deep sub-steps per K tile).
constexpr int BM = 256, BKD = 64, WM = 2, WTM = 128, WTN = 64, TM = WTM / 16;
constexpr int CPR = BKD / 8;                    // 16-byte chunks per K row
constexpr int A_BYTES = BM * BKD * 2;
constexpr int KK = BKD / 32;                     // MFMA sub-steps per K tile
// K-contiguous row r, chunk c -> 16-byte slot (c ^ ((r >> 1) & 7)).
__device__ inline int kslot(int r, int c) { return r * CPR + (c ^ ((r >> 1) & 7)); }
// BN = 256 with 128 x 64 wave tiles (8 waves, 2 x 4), 192 with WTN_ = 48
// (8 waves of 128 x 48, K-contiguous B only) or 128 with WTN_ = 32 (8 waves
// of 128 x 32).  (128-wide tiles on 4 waves of 128 x 64 measured 20-28 %
// slower than on 8 of 128 x 32, e.g. 869 against 1074 TFLOP/s at 2048 x
// 4096 x 4096: with one wave per SIMD the compiler keeps the accumulators in
// AGPRs and copies each through VGPRs on every K tile.)
// (WTN_ = 128, 128 x 128 wave tiles with 256 accumulator registers, one
// wave per SIMD on a 256-wide tile, reads a third less from LDS per MFMA
// but measured slower: 2-3 % with 32x32x16 MFMAs, 30 % with 16x16x32 ones,
// whose accumulators the compiler then moves between register files inside
// the loop; one wave per SIMD also hides less of the K-tile barrier and the
// LDS latency.)
template <int BN_, int WTN_ = WTN>
struct Cfg {
  static constexpr int WTN = WTN_, TN = WTN / 16, NMF = TM * TN, EPITCH = WTN + 8;
  static constexpr int BN = BN_, WN = BN / WTN, NW = WM * WN, NT = NW * 64;
  static constexpr int B_BYTES = BN * BKD * 2, STAGE = A_BYTES + B_BYTES;
  static constexpr int LPA = A_BYTES / 1024 / NW, LPB = B_BYTES / 1024 / NW;  // DMA lines per wave
  static constexpr int BCH = BN / 8;             // 16-byte chunks per row-major B row
  static_assert(LPA * NW * 1024 == A_BYTES && LPB * NW * 1024 == B_BYTES, "DMA lines");
  // the K-tile barrier comes before MFMA XB of the last sub-step
  static constexpr int XB = 8 < NMF - LPA - LPB ? 8 : NMF - LPA - LPB;
  static_assert(XB >= TN - 1, "barrier after the last reads of the stage");
  // the DMA lines after the barrier go out one every DSP MFMAs
  static constexpr int DSP = (NMF - XB) / (LPA + LPB) < 3 ? (NMF - XB) / (LPA + LPB) : 3;
  static_assert(DSP >= 1, "DMA fits in the post-barrier sub-step");
  static_assert(NW * 32 * EPITCH * 4 <= 2 * STAGE, "epilogue staging exceeds LDS");
};
}  // namespace dl

// SWIGLU: B holds the gate rows [0, n) and the up rows [n, 2n) of one
// weight matrix (K-contiguous) and D[m, j] = silu(A B_gate[j]) * (A B_up[j]).
// A 256-wide tile then covers 128 output columns: in the 64 columns of wave
// wn, MFMA tiles 0 and 1 take gate rows j0 + 32 wn .. + 31 and tiles 2 and 3
// the up rows of the same columns, so a lane's accumulators j and j + 2
// hold the gate and up sums of the same output element and the epilogue
// combines them in registers.
template <typename T, bool B_KCONT, int BN_, bool SWIGLU = false, int WTN_ = dl::WTN>
__global__ void __launch_bounds__((dl::Cfg<BN_, WTN_>::NT)) gemm_dl_kernel(const GemmArgs p) {
  using namespace dl;
  using DC = Cfg<BN_, WTN_>;
  constexpr int WTN = DC::WTN, TN = DC::TN, NMF = DC::NMF, EPITCH = DC::EPITCH;
  static_assert(!SWIGLU || (B_KCONT && BN_ == 256), "SwiGLU tiles: K-contiguous B, 256 wide");
  static_assert(B_KCONT || (BN_ / 8) % 16 == 0, "row-major B: the swizzle needs 16-chunk row groups");
  constexpr int BN = DC::BN, WN = DC::WN, STAGE = DC::STAGE, LPA = DC::LPA, LPB = DC::LPB;
  constexpr int NBR = B_KCONT ? 1 : 2;           // LDS reads per B fragment
  constexpr int XB = DC::XB;                     // barrier before this MFMA of the last sub-step
  __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE];

  // Tile rank and K slice: workgroups past tail_start are split-K slices of
  // the tail tiles.
  int rank = blockIdx.x, split = 0;
  const bool partial = rank >= p.tail_start;
  if (partial) {
    const int q = rank - p.tail_start;
    rank = p.tail_start + q / p.splits;
    split = q % p.splits;
  }
  int tm, tn;
  tile_of(rank, p.tiles_m, p.tiles_n, tm, tn);
  const int64_t batch = blockIdx.y;
  // first output column (SwiGLU: 128 output columns per tile)
  const int64_t m0 = static_cast<int64_t>(tm) * BM, n0 = static_cast<int64_t>(tn) * (SWIGLU ? BN / 2 : BN);
  const uint16_t* A = static_cast<const uint16_t*>(p.a) + batch * p.stride_a;
  const uint16_t* B = static_cast<const uint16_t*>(p.b) + batch * p.stride_b;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int lda = static_cast<int>(p.lda), ldb = static_cast<int>(p.ldb);
  const int ksteps_all = static_cast<int>(p.k / BKD);
  const int kt0 = partial ? split * p.kslice : 0;  // first K tile of this workgroup
  const int ksteps = partial ? min(p.kslice, ksteps_all - kt0) : ksteps_all;

  // Buffer ranges: exactly the bytes this tile's rows (columns) span, so the
  // rows of a last, partial tile that lie past M or N read zeros (and are
  // not stored).
  const int64_t arows = min(static_cast<int64_t>(BM), p.m - m0);
  const int64_t brows = min(static_cast<int64_t>(BN), (B_KCONT ? p.n : p.nb) - n0);
  const i32x4 ra = buffer_rsrc(A + m0 * lda, static_cast<uint32_t>(((arows - 1) * lda + p.k) * 2));
  // (SwiGLU: from gate row n0 to up row n + n0 + 127)
  const i32x4 rb = SWIGLU
      ? buffer_rsrc(B + n0 * ldb, static_cast<uint32_t>(((p.n + BN / 2 - 1) * static_cast<int64_t>(ldb) + p.k) * 2))
      : B_KCONT
      ? buffer_rsrc(B + n0 * ldb, static_cast<uint32_t>(((brows - 1) * ldb + p.k) * 2))
      : buffer_rsrc(B + n0, static_cast<uint32_t>(((p.k - 1) * ldb + brows) * 2));
  // Per-lane global byte offsets of this wave's DMA lines (K tile 0).
  uint32_t va[LPA], vb[LPB];
#pragma unroll
  for (int i = 0; i < LPA; ++i) {
    const int s = (wave * LPA + i) * 64 + lane;  // LDS slot filled by this lane
    const int r = s / CPR, c = (s % CPR) ^ ((r >> 1) & 7);
    va[i] = static_cast<uint32_t>(r * lda * 2 + c * 16);
  }
#pragma unroll
  for (int i = 0; i < LPB; ++i) {
    const int s = (wave * LPB + i) * 64 + lane;
    if constexpr (SWIGLU) {
      // LDS row r (tile column) -> weight row: gate j0 + 32 (r / 64) + r % 32
      // for r % 64 < 32, else the matching up row (+ n)
      const int r = s / CPR, c = (s % CPR) ^ ((r >> 1) & 7);
      const int64_t wr = 32 * (r >> 6) + (r & 31) + ((r & 32) ? p.n : 0);
      vb[i] = static_cast<uint32_t>(wr * ldb * 2 + c * 16);
    } else if constexpr (B_KCONT) {
      const int r = s / CPR, c = (s % CPR) ^ ((r >> 1) & 7);
      vb[i] = static_cast<uint32_t>(r * ldb * 2 + c * 16);
    } else {
      const int k = s / DC::BCH, c = (s % DC::BCH) ^ bswz(k);
      vb[i] = static_cast<uint32_t>(k * ldb * 2 + c * 16);
    }
  }
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((SPH_LDS char*)(lds)));
  // Fragment reads.  16x16x32 operands: lane l holds row (column) l % 16 and
  // the 8 K values 8 (l / 16) .. + 7 of the sub-step, one 16-byte chunk of a
  // K-contiguous row: chunk 4 kk + l / 16, whose slot is swizzled by
  // (r >> 1) & 7 = (l % 16 >> 1) & 7 for every tile (tiles start at rows that
  // are multiples of 16), so offset(kk, tile t) = off[kk] + 2048 t.
  const int m16 = lane & 15, g4 = lane >> 4, sw = g4 ^ ((m16 >> 1) & 7);
  int aoff[KK], bkoff[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
    aoff[kk] = (wm * WTM + m16) * (CPR * 16) + ((sw ^ (4 * kk)) << 4);
    bkoff[kk] = A_BYTES + (wn * WTN + m16) * (CPR * 16) + ((sw ^ (4 * kk)) << 4);
  }
  // Row-major B: two transposing reads per fragment.  ds_read_b64_tr_b16
  // has each 16-lane group read a 4 x 16 block (lane e * 4 + q: row e,
  // columns 4q .. 4q + 3) and hands lane m column m of it; group g4 reads K
  // rows 32 kk + 8 g4 + 4 h + e of the fragment's 16 columns.
  int boff[TN];
  {
    const int e = m16 >> 2, q = m16 & 3;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = wn * WTN + j * 16 + 4 * q;
      boff[j] = A_BYTES + (8 * g4 + e) * (BN * 2) + (((n >> 3) ^ bswz(8 * g4 + e)) << 4) + 8 * (q & 1);
    }
  }

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 af[2][TM];
  u32x2 bl[2][TN], bh[2][TN];

// Fragment reads of sub-step KK_ from the stage at byte offset STB_ into
// buffer BUF_: A tile I_; B fragment read X_ (K-contiguous: fragment X_;
// row-major: fragment X_ / 2, half X_ % 2).
#define SPH_DL_READ_A(BUF_, I_, STB_, KK_)                                                  \
  af[BUF_][I_] = *reinterpret_cast<const u32x4*>(lds + (STB_) + aoff[KK_] + (I_) * 2048)
#define SPH_DL_READ_B(BUF_, X_, STB_, KK_)                                                  \
  do {                                                                                      \
    if constexpr (B_KCONT) {                                                                \
      const u32x4 v_ =                                                                      \
          *reinterpret_cast<const u32x4*>(lds + (STB_) + bkoff[KK_] + (X_) * 2048);         \
      bl[BUF_][X_] = u32x2{v_[0], v_[1]};                                                   \
      bh[BUF_][X_] = u32x2{v_[2], v_[3]};                                                   \
    } else {                                                                                \
      const int j_ = (X_) >> 1, h_ = (X_) & 1;                                              \
      const SPH_LDS char* p_ = (const SPH_LDS char*)(lds + (STB_)) + boff[j_] +             \
                               ((KK_) * 32 + 4 * h_) * (BN * 2);                            \
      const u32x2 v_ = __builtin_bit_cast(                                                  \
          u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((SPH_LDS s16x4*)(p_)));            \
      if (h_) bh[BUF_][j_] = v_;                                                            \
      else bl[BUF_][j_] = v_;                                                               \
    }                                                                                       \
  } while (0)
// DMA line LINE_ (A lines first, then B) of K tile T_ into stage SL_ & 1.
#define SPH_DL_DMA(T_, SL_, LINE_)                                                          \
  do {                                                                                      \
    const int t_ = (T_), l_ = (LINE_);                                                      \
    const uint32_t sb_ = lds_base + ((SL_) & 1) * STAGE;                                    \
    if (l_ < LPA)                                                                           \
      dma16(ra, __builtin_amdgcn_readfirstlane(sb_ + (wave * LPA + l_) * 1024), va[l_],     \
            __builtin_amdgcn_readfirstlane((kt0 + t_) * BKD * 2));                          \
    else                                                                                    \
      dma16(rb, __builtin_amdgcn_readfirstlane(sb_ + A_BYTES + (wave * LPB + l_ - LPA) * 1024), \
            vb[l_ - LPA],                                                                   \
            __builtin_amdgcn_readfirstlane(B_KCONT ? (kt0 + t_) * BKD * 2                   \
                                                   : (kt0 + t_) * BKD * ldb * 2));          \
  } while (0)

  // Prologue: K tiles 0 and 1 in flight; wait for tile 0; the fragments of
  // its first sub-step.
#pragma unroll
  for (int l = 0; l < LPA + LPB; ++l) SPH_DL_DMA(0, 0, l);
  if (ksteps > 1) {
#pragma unroll
    for (int l = 0; l < LPA + LPB; ++l) SPH_DL_DMA(1, 1, l);
    wait_vmcnt<LPA + LPB>();
  } else {
    wait_vmcnt<0>();
  }
  __syncthreads();
#pragma unroll
  for (int x = 0; x < TN * NBR; ++x) SPH_DL_READ_B(0, x, 0, 0);
#pragma unroll
  for (int i = 0; i < TM; ++i) SPH_DL_READ_A(0, i, 0, 0);

  // Sub-step kk: MFMA x = (A tile x / TN, B fragment x % TN, or TN - 1 -
  // x % TN for odd A tiles).  Its reads of
  // the next sub-step's fragments: the B reads first (the next sub-step's
  // first MFMAs need all of B), each A tile right after the last MFMA that
  // uses this sub-step's A tile of the same index (so the two can share
  // registers).  Before MFMA XB of the last sub-step a wave waits for its own
  // DMA of the next K tile and its own LDS reads, then joins the barrier;
  // after it the sub-step reads the next tile's fragments and issues the DMA
  // of the tile after next into the stage just vacated.  Past the last tile
  // the DMA re-loads the last tile and the fragment reads fetch values nobody
  // uses, so the loop has no branches.
  for (int ks = 0; ks < ksteps; ++ks) {
    const int cs = (ks & 1) * STAGE, ns = ((ks + 1) & 1) * STAGE;
    const int tnext = ks + 2 < ksteps ? ks + 2 : ksteps - 1;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const bool lastk = kk == KK - 1;
      const int nst = lastk ? ns : cs;           // stage of the next sub-step
      const int nkk = lastk ? 0 : kk + 1;        // and its index
      const int x0 = lastk ? XB : 0;             // first slot of the B reads
#pragma unroll
      for (int x = 0; x < NMF; ++x) {
        // A tile i; B fragments in alternating directions, so consecutive
        // MFMAs across a tile boundary share their B operand (~1 % faster)
        const int i = x / TN, j = (x / TN) & 1 ? TN - 1 - x % TN : x % TN;
        if (lastk && x == XB) {
          wait_vmcnt<0>();
          wait_lgkmcnt0();
          __syncthreads();
        }
        {
          const u32x4 b_ = __builtin_shufflevector(bl[kk & 1][j], bh[kk & 1][j], 0, 1, 2, 3);
          acc[i][j] = mfma16<T>(af[kk & 1][i], b_, acc[i][j]);
        }
        if (x >= x0 && x - x0 < TN * NBR) SPH_DL_READ_B((kk + 1) & 1, x - x0, nst, nkk);
#pragma unroll
        for (int ii = 0; ii < TM; ++ii) {
          // after this sub-step's last use of A tile ii (the last sub-step
          // shifts the reads past the barrier)
          const int last_use = ii * TN + TN - 1;
          const int at = lastk ? min(NMF - 1, last_use + XB - (TN - 1)) : last_use;
          if (x == at) SPH_DL_READ_A((kk + 1) & 1, ii, nst, nkk);
        }
        if (lastk && x >= XB && (x - XB) % DC::DSP == 0 && (x - XB) / DC::DSP < LPA + LPB)
          SPH_DL_DMA(tnext, ks, (x - XB) / DC::DSP);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
#undef SPH_DL_READ_A
#undef SPH_DL_READ_B
#undef SPH_DL_DMA

  // Epilogue (LDS reused as fp32 slabs once every DMA has landed).  16x16
  // accumulator r of lane l: row 4 (l / 16) + r, column l % 16 of its tile.
  wait_vmcnt<0>();
  if (partial) {
    // split-K slice: the raw fp32 tile, element (r, c) at r * BN + c
    float* W = p.part + (static_cast<int64_t>(rank - p.tail_start) * p.splits + split) * (BM * BN);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = wm * WTM + i * 16 + 4 * g4 + r;
          W[row * BN + wn * WTN + j * 16 + m16] = acc[i][j][r];
        }
    return;
  }
  __syncthreads();
  T* D = static_cast<T*>(p.d) + batch * p.stride_d;
  const T* C = p.c ? static_cast<const T*>(p.c) + batch * p.stride_c : nullptr;
  float* slab = reinterpret_cast<float*>(lds) + wave * (32 * EPITCH);
  const int64_t row0 = m0 + wm * WTM;
  auto chunks = [&](auto epi_, auto use_c_) {
    constexpr int E = decltype(epi_)::value;
    constexpr bool UC = decltype(use_c_)::value;
    if constexpr (SWIGLU) {
      // silu(gate) * up per element, 32 output columns per wave
      static_assert(TN == 4, "gate / up tile pairs");
      constexpr int SP = 32 + 8;
      const int64_t colw = n0 + wn * 32;
#pragma unroll
      for (int i2 = 0; i2 < TM / 2; ++i2) {
#pragma unroll
        for (int ii = 0; ii < 2; ++ii)
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              slab[(ii * 16 + 4 * g4 + r) * SP + j * 16 + m16] =
                  silu(acc[2 * i2 + ii][j][r]) * acc[2 * i2 + ii][j + 2][r];
        __syncthreads();
        store_slab_impl<T, E, UC, 32, SP>(p, slab, D, C, row0 + i2 * 32, colw, lane);
        __syncthreads();
      }
    } else {
      const int64_t colw = n0 + wn * WTN;
#pragma unroll
      for (int i2 = 0; i2 < TM / 2; ++i2) {
#pragma unroll
        for (int ii = 0; ii < 2; ++ii)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              slab[(ii * 16 + 4 * g4 + r) * EPITCH + j * 16 + m16] = acc[2 * i2 + ii][j][r];
        __syncthreads();
        store_slab_impl<T, E, UC, WTN, EPITCH>(p, slab, D, C, row0 + i2 * 32, colw, lane);
        __syncthreads();
      }
    }
  };
  epi_dispatch(p, C, chunks);
}

// Sums the split-K slices of one tail tile and applies the epilogue: one
// workgroup per (tail tile, 1024 output elements); each thread takes 4
// consecutive output columns of one row (16-byte reads of every slice).
// SWIGLU: output column oc of the tile is silu(gate) * up with the gate sum
// at tile column 64 (oc / 32) + oc % 32 and the up sum 32 columns further.

template <typename T, int BN, bool SWIGLU>
__global__ void __launch_bounds__(256) gemm_splitk_reduce(const GemmArgs p) {
  constexpr int OUTN = SWIGLU ? BN / 2 : BN;   // output columns per tile
  constexpr int PER_WG = 1024;                  // outputs per workgroup
  const int t = blockIdx.x;                     // tail tile
  const int e = blockIdx.y * PER_WG + threadIdx.x * 4;
  const int r = e / OUTN, oc = e % OUTN;
  int tm, tn;
  tile_of(p.tail_start + t, p.tiles_m, p.tiles_n, tm, tn);
  const int64_t row = static_cast<int64_t>(tm) * dl::BM + r;
  const int64_t col = static_cast<int64_t>(tn) * OUTN + oc;
  if (row >= p.m || col >= p.n) return;
  const float* W = p.part + static_cast<int64_t>(t) * p.splits * (dl::BM * BN) + r * BN;
  float v[4] = {0.f, 0.f, 0.f, 0.f}, u[4] = {0.f, 0.f, 0.f, 0.f};
  const int cg = SWIGLU ? 64 * (oc / 32) + oc % 32 : oc;
  for (int sp = 0; sp < p.splits; ++sp) {
    const float* Ws = W + static_cast<int64_t>(sp) * (dl::BM * BN);
    const f32x4 a = *reinterpret_cast<const f32x4*>(Ws + cg);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += a[i];
    if constexpr (SWIGLU) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(Ws + cg + 32);
#pragma unroll
      for (int i = 0; i < 4; ++i) u[i] += b[i];
    }
  }
  T* D = static_cast<T*>(p.d);
  float out[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float x;
    if constexpr (SWIGLU) {
      x = silu(v[i]) * u[i];
    } else {
      x = p.alpha * v[i];
      if (p.c != nullptr && p.beta != 0.f && col + i < p.n)
        x += p.beta * Num<T>::to_f(static_cast<const T*>(p.c)[row * p.ldc_row + (col + i) * p.ldc_col]);
      if (p.epilogue == SPH_EPI_RELU) x = fmaxf(x, 0.f);
      else if (p.epilogue == SPH_EPI_GELU) x = gelu_erf(x);
      else if (p.epilogue == SPH_EPI_SILU) x = silu(x);
    }
    out[i] = x;
  }
  if (col + 4 > p.n) {  // last columns of a ragged N
    for (int i = 0; i < 4 && col + i < p.n; ++i) D[row * p.ldd + col + i] = Num<T>::from_f(out[i]);
    return;
  }
  u32x2 w;
  w[0] = static_cast<uint32_t>(__builtin_bit_cast(uint16_t, Num<T>::from_f(out[0]))) |
         (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, Num<T>::from_f(out[1]))) << 16);
  w[1] = static_cast<uint32_t>(__builtin_bit_cast(uint16_t, Num<T>::from_f(out[2]))) |
         (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, Num<T>::from_f(out[3]))) << 16);
  typedef u32x2 u32x2_any __attribute__((aligned(2)));
  *reinterpret_cast<u32x2_any*>(D + row * p.ldd + col) = w;
}

// ---------------------------------------------------------------------------
// Short-K products (K = 64 or 128; e.g. attention scores Q K^T with head
// dim 128): at 2 M N K FLOP against 2 M N bytes of output they are bound by
// memory.  Design:
//   * 128x128 tiles on 4 waves (64x64 each); the whole K range is one LDS
//     stage (64 KB at K = 128), so two workgroups share a CU and one's
//     operand loads overlap the other's MFMAs and stores.  (A persistent
//     one-workgroup-per-CU variant with a two-stage operand ring, with and
//     without producer/consumer wave roles, measured slower: its DMA keeps
//     at most one tile in flight per CU, and under the output stream the
//     load latency, not bandwidth, then sets the pace.  A variant with A's
//     MFMA fragments loaded straight from memory into registers and only B
//     in LDS (32 KB: three workgroups per CU) measured 86 us against 77.5
//     on the c2 bmm shape.)
//   * Operands arrive by direct global->LDS DMA as in the whole-tile kernel
//     (one 64-deep K block after another, same layouts; row-major B rows
//     are 256 bytes here and use chunk slot c ^ 4 (k & 3)).
//   * The MFMAs take B as the first operand, so each lane's accumulators
//     hold 4 consecutive output columns of one row: converted to T they are
//     8-byte LDS writes into a per-wave 64 x 64 slab (16-byte chunk c of row
//     m at slot c ^ ((m >> 1) & 7)), read back as whole 128-byte rows and
//     stored with 16-byte stores.
//   * Plain products only (alpha = 1, no C, no activation): D rounds each
//     fp32 sum once.
// ---------------------------------------------------------------------------
namespace sk {
constexpr int BM = 128, BN = 128, WM = 2, WN = 2, NW = WM * WN, NT = NW * 64;
constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 32, TN = WTN / 32;
constexpr int KB = 64;                           // K block (one A and one B block per 64 K)
constexpr int A_BLK = BM * KB * 2, B_BLK = BN * KB * 2;  // 16 KB each
constexpr int LPW = A_BLK / 1024 / NW;           // DMA lines per wave per block
constexpr int SLAB = WTM * WTN * 2;              // per-wave output slab (bytes)
static_assert(LPW * NW * 1024 == A_BLK, "DMA lines");
__device__ inline int aslot(int r, int c) { return r * 8 + (c ^ ((r >> 1) & 7)); }
}  // namespace sk

template <typename T, bool B_KCONT, int KT>
__global__ void __launch_bounds__(sk::NT) gemm_shortk_kernel(const GemmArgs p) {
  using namespace sk;
  constexpr int OPS = KT * (A_BLK + B_BLK);
  static_assert(NW * SLAB <= OPS, "slab fits in the operand space");
  __shared__ __attribute__((aligned(1024))) char lds[OPS];
  int tm, tn;
  tile_of(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
  const int64_t batch = blockIdx.y;
  const int64_t m0 = static_cast<int64_t>(tm) * BM, n0 = static_cast<int64_t>(tn) * BN;
  const uint16_t* A = static_cast<const uint16_t*>(p.a) + batch * p.stride_a;
  const uint16_t* B = static_cast<const uint16_t*>(p.b) + batch * p.stride_b;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int lda = static_cast<int>(p.lda), ldb = static_cast<int>(p.ldb);

  const i32x4 ra = buffer_rsrc(A + m0 * lda, static_cast<uint32_t>(((BM - 1) * static_cast<int64_t>(lda) + p.k) * 2));
  const i32x4 rb = B_KCONT
      ? buffer_rsrc(B + n0 * ldb, static_cast<uint32_t>(((BN - 1) * static_cast<int64_t>(ldb) + p.k) * 2))
      : buffer_rsrc(B + n0, static_cast<uint32_t>(((p.k - 1) * ldb + BN) * 2));
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((SPH_LDS char*)(lds)));
#pragma unroll
  for (int kb = 0; kb < KT; ++kb) {
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int line = wave * LPW + i;
      const int s = line * 64 + lane;
      const int r = s >> 3, c = (s & 7) ^ ((r >> 1) & 7);
      dma16(ra, __builtin_amdgcn_readfirstlane(lds_base + kb * A_BLK + line * 1024),
            static_cast<uint32_t>(r * lda * 2 + c * 16), __builtin_amdgcn_readfirstlane(kb * KB * 2));
      uint32_t vb;
      if constexpr (B_KCONT) {
        vb = static_cast<uint32_t>(r * ldb * 2 + c * 16);
      } else {
        const int k = s >> 4, cb = (s & 15) ^ (4 * (k & 3));
        vb = static_cast<uint32_t>(k * ldb * 2 + cb * 16);
      }
      dma16(rb, __builtin_amdgcn_readfirstlane(lds_base + KT * A_BLK + kb * B_BLK + line * 1024), vb,
            __builtin_amdgcn_readfirstlane(B_KCONT ? kb * KB * 2 : kb * KB * ldb * 2));
    }
  }
  wait_vmcnt<0>();
  __syncthreads();

  const int row_in = lane & 31, khalf = lane >> 5;
  const int g = lane >> 4, jj = lane & 15, e = jj >> 2, q = jj & 3;
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
#pragma unroll
  for (int kb = 0; kb < KT; ++kb) {
    const char* sa = lds + kb * A_BLK;
    const char* sb = lds + KT * A_BLK + kb * B_BLK;
#pragma unroll
    for (int kk = 0; kk < KB / 16; ++kk) {
      u32x4 af[TM], bf[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        af[i] = *reinterpret_cast<const u32x4*>(sa + aslot(wm * WTM + i * 32 + row_in, kk * 2 + khalf) * 16);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (B_KCONT) {
          bf[j] = *reinterpret_cast<const u32x4*>(sb + aslot(wn * WTN + j * 32 + row_in, kk * 2 + khalf) * 16);
        } else {
          const int n = wn * WTN + j * 32 + 16 * (g & 1) + 4 * q;
          const int k = kk * 16 + 8 * (g >> 1) + e;
          const SPH_LDS char* p0 =
              (const SPH_LDS char*)(sb) + k * (BN * 2) + (((n >> 3) ^ (4 * e)) << 4) + 8 * (q & 1);
          const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((SPH_LDS s16x4*)(p0)));
          const u32x2 hi = __builtin_bit_cast(
              u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((SPH_LDS s16x4*)(p0 + 4 * BN * 2)));
          bf[j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3);
        }
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mfma32<T>(bf[j], af[i], acc[i][j]);
    }
  }
  // acc[i][j][r]: row m = i*32 + lane%32, columns n = j*32 + 8*(r/4) + 4*(lane/32) + r%4
  __syncthreads();
  char* slab = lds + wave * SLAB;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = i * 32 + row_in;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int n = j * 32 + 8 * rg + 4 * khalf;
        uint32_t w[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint16_t lo = __builtin_bit_cast(uint16_t, Num<T>::from_f(acc[i][j][4 * rg + 2 * h]));
          const uint16_t hi = __builtin_bit_cast(uint16_t, Num<T>::from_f(acc[i][j][4 * rg + 2 * h + 1]));
          w[h] = static_cast<uint32_t>(lo) | (static_cast<uint32_t>(hi) << 16);
        }
        const int c = n >> 3;
        *reinterpret_cast<u32x2*>(slab + (m * 8 + (c ^ ((m >> 1) & 7))) * 16 + (n & 7) * 2) =
            u32x2{w[0], w[1]};
      }
  }
  // The slab belongs to this wave alone; a wave's LDS accesses run in order.
  // The output is written once and not read back by this kernel: streaming
  // (non-temporal) stores, 14 % faster than plain ones on the attention-
  // score shape (32 x 2048 x 2048 from K = 128).
  T* D = static_cast<T*>(p.d) + batch * p.stride_d;
#pragma unroll
  for (int it = 0; it < WTM / 8; ++it) {
    const int m = it * 8 + (lane >> 3), c = lane & 7;
    const u32x4 v = *reinterpret_cast<const u32x4*>(slab + (m * 8 + (c ^ ((m >> 1) & 7))) * 16);
    __builtin_nontemporal_store(
        v, reinterpret_cast<u32x4*>(D + (m0 + wm * WTM + m) * p.ldd + n0 + wn * WTN + c * 8));
  }
}

// ---------------------------------------------------------------------------
// Short-K products over many tiles (the attention scores of a whole batch):
// a persistent form of the kernel above, one workgroup of 4 waves (64x64
// each) per CU, walking a contiguous run of the (batch entry, tile row,
// tile column) sequence of 128x128 tiles.
//   * The A row panel of the current (batch entry, tile row) stays in LDS
//     while the workgroup walks that row's tile columns, so a tile streams
//     only its B block: half the operand bytes of the one-shot kernel.
//   * B blocks go through a three-stage LDS ring: while tile i computes,
//     tiles i+1 and i+2 are in flight (issued one and two tiles earlier).
//   * Results leave through a per-wave 32 x 64 slab (two halves per tile)
//     as streaming 16-byte stores of whole 128-byte rows that the loop never
//     waits for: vector memory counts return in issue order, so waiting for
//     an older block's DMA leaves the stores issued after it in flight.
//   * Consecutive workgroups of one XCD (dispatch is round-robin over the 8
//     XCDs) take consecutive runs, so one batch entry's B panel is fetched
//     into one XCD's L2 and re-read from there by its tile rows.
//   * The tile position advances by a cursor (no 64-bit divisions in the
//     loop) and each tile's first MFMAs take a zero accumulator operand.
// A new A panel (a run crossing into the next tile row) is loaded after
// every wave has finished the previous tile: one exposed load per switch,
// at most a few per workgroup.
// Measured on MI355X (attention-score shape 32 x 2048 x 2048 from K = 128,
// alternating on one box): 67.5-70 us against 79-81 for the one-shot
// kernel.  Not kept: 8 waves of 64x32 (64-byte row stores) 93-95 us; 8
// waves of 32x64, 69.6; 256-row tiles on 8 waves with a two-stage ring,
// 76.5 against 74.3 on a slower box; the same kernel with 64-bit tile
// divisions and zeroed accumulators, 75; tile i-1's slab epilogue and
// stores spread between tile i's MFMA sub-steps, 73-74 against 69-71.
// ---------------------------------------------------------------------------
namespace skr {
constexpr int NSTG = 3;                               // B stages
// Wave layout WM x WN over the 128x128 tile.
template <int WM_, int WN_>
struct L {
  static constexpr int WM = WM_, WN = WN_, NW = WM * WN, NT = NW * 64;
  static constexpr int WTM = sk::BM / WM, WTN = sk::BN / WN, TM = WTM / 32, TN = WTN / 32;
  static constexpr int CPR = WTN * 2 / 16;            // 16-byte chunks per slab row
  static constexpr int RPS = 1024 / (WTN * 2);        // slab rows per 16-byte store instruction
  static constexpr int SLAB = 32 * WTN * 2;           // per-wave slab: 32 rows of the wave tile
  static constexpr int STORES = TM * 32 / RPS;        // stores per wave per tile
  static constexpr int LPW = sk::A_BLK / 1024 / NW;   // DMA lines per wave per 64-deep block
  static_assert(LPW * NW * 1024 == sk::A_BLK && (CPR & (CPR - 1)) == 0, "wave layout");
  // slab row m, chunk c -> 16-byte slot
  __device__ static int sslot(int m, int c) { return m * CPR + (c ^ ((m >> 1) & (CPR - 1))); }
};
// Position (batch entry, tile row, tile column) in the tile sequence.
struct Cursor {
  int b, tm, tn;
  __device__ void next(int tiles_m, int tiles_n) {
    if (++tn == tiles_n) {
      tn = 0;
      if (++tm == tiles_m) tm = 0, ++b;
    }
  }
};
}  // namespace skr

template <typename T, bool B_KCONT, int KT, int WM_, int WN_>
__global__ void __launch_bounds__((skr::L<WM_, WN_>::NT)) gemm_shortk_ring_kernel(const GemmArgs p) {
  using sk::A_BLK;
  using sk::B_BLK;
  using sk::BM;
  using sk::BN;
  using sk::KB;
  using sk::aslot;
  using skr::Cursor;
  using skr::NSTG;
  using W = skr::L<WM_, WN_>;
  constexpr int WN = W::WN, WTM = W::WTM, WTN = W::WTN, TM = W::TM, TN = W::TN;
  constexpr int NW = W::NW, LPW = W::LPW, STORES = W::STORES, CPR = W::CPR, RPS = W::RPS;
  constexpr int A_PANEL = KT * A_BLK, B_TILE = KT * B_BLK;
  constexpr int LB = KT * LPW;                     // DMA lines per wave per B block (= per A panel)
  constexpr int SLAB_OFF = A_PANEL + NSTG * B_TILE;
  __shared__ __attribute__((aligned(1024))) char lds[SLAB_OFF + NW * W::SLAB];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int lda = static_cast<int>(p.lda), ldb = static_cast<int>(p.ldb);
  const int tiles_m = p.tiles_m, tiles_n = p.tiles_n;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((SPH_LDS char*)(lds)));

  // This workgroup's run [t0, t0 + n) of the tile sequence.
  const int64_t total = p.batches * tiles_m * tiles_n;
  const int G = static_cast<int>(gridDim.x);
  int slot = static_cast<int>(blockIdx.x);
  if ((G & 7) == 0) slot = (slot & 7) * (G >> 3) + (slot >> 3);
  const int64_t t0 = total * slot / G;
  const int n = static_cast<int>(total * (slot + 1) / G - t0);
  if (n <= 0) return;
  Cursor cur;  // tile i
  {
    const int64_t u = t0 / tiles_n;
    cur.tn = static_cast<int>(t0 - u * tiles_n);
    cur.b = static_cast<int>(u / tiles_m);
    cur.tm = static_cast<int>(u - static_cast<int64_t>(cur.b) * tiles_m);
  }

  // Per-lane byte offsets of this wave's DMA lines within a 64-deep K block.
  uint32_t va[LPW], vb[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int s = (wave * LPW + i) * 64 + lane;
    const int r = s >> 3, c = (s & 7) ^ ((r >> 1) & 7);
    va[i] = static_cast<uint32_t>(r * lda * 2 + c * 16);
    if constexpr (B_KCONT) {
      vb[i] = static_cast<uint32_t>(r * ldb * 2 + c * 16);
    } else {
      const int k = s >> 4, cb = (s & 15) ^ (4 * (k & 3));
      vb[i] = static_cast<uint32_t>(k * ldb * 2 + cb * 16);
    }
  }
  const uint16_t* const A0 = static_cast<const uint16_t*>(p.a);
  const uint16_t* const B0 = static_cast<const uint16_t*>(p.b);
  // A row panel of the cursor's (batch entry, tile row) into the panel slot.
  auto dma_a = [&](const Cursor& c) {
    const i32x4 ra = buffer_rsrc(A0 + c.b * p.stride_a + static_cast<int64_t>(c.tm) * BM * p.lda,
                                 static_cast<uint32_t>(((BM - 1) * static_cast<int64_t>(lda) + p.k) * 2));
#pragma unroll
    for (int kb = 0; kb < KT; ++kb)
#pragma unroll
      for (int i = 0; i < LPW; ++i)
        dma16(ra, __builtin_amdgcn_readfirstlane(lds_base + kb * A_BLK + (wave * LPW + i) * 1024), va[i],
              __builtin_amdgcn_readfirstlane(kb * KB * 2));
  };
  // B block of the cursor's tile into ring stage st.
  auto dma_b = [&](const Cursor& c, int st) {
    const uint16_t* B = B0 + c.b * p.stride_b;
    const i32x4 rb = B_KCONT
        ? buffer_rsrc(B + static_cast<int64_t>(c.tn) * BN * p.ldb,
                      static_cast<uint32_t>(((BN - 1) * static_cast<int64_t>(ldb) + p.k) * 2))
        : buffer_rsrc(B + static_cast<int64_t>(c.tn) * BN, static_cast<uint32_t>(((p.k - 1) * ldb + BN) * 2));
#pragma unroll
    for (int kb = 0; kb < KT; ++kb)
#pragma unroll
      for (int i = 0; i < LPW; ++i)
        dma16(rb,
              __builtin_amdgcn_readfirstlane(lds_base + A_PANEL + st * B_TILE + kb * B_BLK +
                                             (wave * LPW + i) * 1024),
              vb[i], __builtin_amdgcn_readfirstlane(B_KCONT ? kb * KB * 2 : kb * KB * ldb * 2));
  };

  Cursor ahead = cur;  // tile i + 2 once the loop runs
  dma_a(cur);
  dma_b(ahead, 0);
  ahead.next(tiles_m, tiles_n);
  if (n > 1) dma_b(ahead, 1);
  ahead.next(tiles_m, tiles_n);

  const int row_in = lane & 31, khalf = lane >> 5;
  const int g = lane >> 4, jj = lane & 15, e = jj >> 2, q = jj & 3;
  char* const slab = lds + SLAB_OFF + wave * W::SLAB;
  T* const D0 = static_cast<T*>(p.d);
  bool reloaded = false;  // the previous tile loaded a new A panel
  for (int i = 0; i < n; ++i) {
    const bool sw = i > 0 && cur.tn == 0;  // tile i starts a new tile row
    // B block i (and everything issued before it) has landed.  Issued
    // after it: the stores of tiles i-2 and i-1, B block i+1 unless i is
    // the last tile, and an A panel if tile i-1 switched rows; waiting for
    // fewer than that many waits longer, never shorter.
    if (i == 0) {
      wait_vmcnt<0>();
    } else if (i == 1) {
      wait_vmcnt<STORES>();
    } else if (!reloaded && i + 1 < n) {
      wait_vmcnt<2 * STORES + LB>();
    } else {
      wait_vmcnt<2 * STORES>();
    }
    // Past this barrier every wave is done with tile i-1: its ring stage
    // and, on a row switch, the A panel may be refilled.
    __syncthreads();
    if (sw) dma_a(cur);
    if (i + 2 < n) {
      dma_b(ahead, (i + 2) % NSTG);
      ahead.next(tiles_m, tiles_n);
    }
    if (sw) {
      if (i + 2 < n) wait_vmcnt<LB>();
      else wait_vmcnt<0>();
      __syncthreads();
    }
    reloaded = sw;

    const char* sb = lds + A_PANEL + (i % NSTG) * B_TILE;
    f32x16 acc[TM][TN];
#pragma unroll
    for (int kb = 0; kb < KT; ++kb) {
      const char* sa = lds + kb * A_BLK;
      const char* sbk = sb + kb * B_BLK;
#pragma unroll
      for (int kk = 0; kk < KB / 16; ++kk) {
        u32x4 af[TM], bf[TN];
#pragma unroll
        for (int a = 0; a < TM; ++a)
          af[a] = *reinterpret_cast<const u32x4*>(sa + aslot(wm * WTM + a * 32 + row_in, kk * 2 + khalf) * 16);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if constexpr (B_KCONT) {
            bf[j] = *reinterpret_cast<const u32x4*>(sbk + aslot(wn * WTN + j * 32 + row_in, kk * 2 + khalf) * 16);
          } else {
            const int nn = wn * WTN + j * 32 + 16 * (g & 1) + 4 * q;
            const int k = kk * 16 + 8 * (g >> 1) + e;
            const SPH_LDS char* p0 =
                (const SPH_LDS char*)(sbk) + k * (BN * 2) + (((nn >> 3) ^ (4 * e)) << 4) + 8 * (q & 1);
            const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((SPH_LDS s16x4*)(p0)));
            const u32x2 hi = __builtin_bit_cast(
                u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((SPH_LDS s16x4*)(p0 + 4 * BN * 2)));
            bf[j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3);
          }
        }
        // (the first sub-step starts from a zero accumulator operand)
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[a][j] = mfma32<T>(bf[j], af[a], kb == 0 && kk == 0 ? f32x16{} : acc[a][j]);
      }
    }
    // acc[a][j][r]: row a*32 + lane%32, column j*32 + 8*(r/4) + 4*(lane/32) + r%4.
    // Each 32-row block goes through the wave's own slab: 8-byte writes,
    // 16-byte reads of whole slab rows, streaming stores.
    T* D = D0 + cur.b * p.stride_d + (static_cast<int64_t>(cur.tm) * BM + wm * WTM) * p.ldd +
           static_cast<int64_t>(cur.tn) * BN + wn * WTN;
#pragma unroll
    for (int a = 0; a < TM; ++a) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          uint32_t w[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const uint16_t lo = __builtin_bit_cast(uint16_t, Num<T>::from_f(acc[a][j][4 * rg + 2 * h]));
            const uint16_t hi = __builtin_bit_cast(uint16_t, Num<T>::from_f(acc[a][j][4 * rg + 2 * h + 1]));
            w[h] = static_cast<uint32_t>(lo) | (static_cast<uint32_t>(hi) << 16);
          }
          *reinterpret_cast<u32x2*>(slab + W::sslot(row_in, j * 4 + rg) * 16 + khalf * 8) = u32x2{w[0], w[1]};
        }
#pragma unroll
      for (int it = 0; it < 32 / RPS; ++it) {
        const int m = it * RPS + lane / CPR, c = lane % CPR;
        const u32x4 v = *reinterpret_cast<const u32x4*>(slab + W::sslot(m, c) * 16);
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(D + (a * 32 + m) * p.ldd + c * 8));
      }
    }
    cur.next(tiles_m, tiles_n);
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
// The direct-load kernel addresses a tile's operand rows with 32-bit buffer
// offsets: every byte it may touch must lie within 2^31 of the tile origin.
inline bool dl_fits(const GemmArgs& p, bool b_kcont, int bn) {
  constexpr int64_t kLim = (1LL << 31) - 1;
  if (p.lda > kLim / 2 || p.ldb > kLim / 2) return false;
  const int64_t a_bytes = ((dl::BM - 1) * p.lda + p.k) * 2;
  const int64_t b_bytes = b_kcont ? ((bn - 1) * p.ldb + p.k) * 2 : ((p.k - 1) * p.ldb + bn) * 2;
  return a_bytes < kLim && b_bytes < kLim;
}

constexpr int64_t kNumCUs = 256;  // MI355X compute units

// Split-K for the last, partial round of 256-wide tiles (batch 1): when
// `tiles` is not a multiple of the CU count, the tail tiles would run as a
// round of their own on a few CUs.  Each tail tile is split into up to 8
// K slices (enough to fill the CUs; K >= 2048, so a slice keeps >= 4 K
// tiles) whose fp32 partial tiles a reduce kernel sums.  A tail of 0 (e.g.
// 4096^3) takes no split.  Measured on one MI355X: the c4 decoder layer
// (M = 2048: gate/up 800 tiles, O and down 128 tiles) 1.143 -> 1.037 ms.
struct SplitPlan {
  int splits = 1, kslice = 0;
  int64_t tail_start = 0, bytes = 0;
};
inline SplitPlan splitk_plan(int64_t tiles, int64_t ksteps, int bn) {
  SplitPlan pl;
  pl.tail_start = tiles;
  if (tiles <= 0 || tiles >= (1LL << 30) || ksteps < 32) return pl;
  const int64_t full = tiles / kNumCUs * kNumCUs, tail = tiles - full;
  if (tail == 0) return pl;
  int64_t sp = kNumCUs / tail;
  sp = sp < 8 ? sp : 8;
  if (sp < 2) return pl;
  const int64_t kslice = ceil_div(ksteps, sp);
  sp = ceil_div(ksteps, kslice);  // every slice non-empty
  if (sp < 2) return pl;
  pl.splits = static_cast<int>(sp);
  pl.kslice = static_cast<int>(kslice);
  pl.tail_start = full;
  pl.bytes = tail * sp * dl::BM * bn * 4;
  return pl;
}

// Time model of the direct-load kernel, fitted to fp16 runs on one MI355X
// (us): a round of 256 x 256 tiles (one per CU) takes ~12 us + 22.4 ns per
// K column (104 us at K = 4096, 299 us at K = 12800); a split-K tail round
// the time of its K slice plus ~4 us and the fp32 partials' write and
// reduce at ~4.2 TB/s (~20 us for the 128 tiles x 2 slices of the c4 O and
// down shapes); a round of 128-wide tiles (8 waves of 128 x 32, half the
// MFMAs per K tile, so less time to cover each tile's loads) 0.62 of a
// 256-wide round with its operands in the caches but 0.78 with operands
// from HBM, as a model layer's weights are (2048 x 4096 x 4096 + residual:
// 65 us hot, 86 us cold, against 76 / 80 us split along K; a cold 256-wide
// round at K = 4096: 109 us).  The model takes the cold figure.
inline double dl_round_us(int64_t k) { return 12.0 + 0.0224 * static_cast<double>(k); }
inline double dl_est128(int64_t tiles128, int64_t k) {
  return static_cast<double>(ceil_div(tiles128, kNumCUs)) * 0.78 * dl_round_us(k);
}
inline double dl_est256(int64_t tiles256, int64_t k) {
  return static_cast<double>(ceil_div(tiles256, kNumCUs)) * dl_round_us(k);
}

// The split plan for `tiles` 256-wide tiles (batch 1, N % 256 == 0) where
// the model puts it ahead of whole rounds of 256- and of 128-wide tiles;
// else a plan of one split (no workspace).
inline double splitk_us(const SplitPlan& pl, int64_t k) {
  return static_cast<double>(pl.tail_start / kNumCUs) * dl_round_us(k) +
         dl_round_us(static_cast<int64_t>(pl.kslice) * dl::BKD) + 4.0 +
         static_cast<double>(pl.bytes) / 4.2e6;
}
inline SplitPlan splitk_choice(int64_t tiles, int64_t k) {
  const SplitPlan pl = splitk_plan(tiles, k / dl::BKD, 256);
  if (pl.splits <= 1) return pl;
  const double est = splitk_us(pl, k);
  if (est < dl_est256(tiles, k) && est < dl_est128(2 * tiles, k)) return pl;
  SplitPlan none;
  none.tail_start = tiles;
  return none;
}

// The direct-load kernel's tile width (kind 256, 192 or 128; 0: none fits)
// for a call, its split plan and the modelled time.
struct DlChoice {
  int kind = 0;
  double us = 0;
  SplitPlan split;
};
inline DlChoice dl_choice(const GemmArgs& p, int64_t batch, bool b_kcont) {
  DlChoice c;
  const int64_t tm = ceil_div(p.m, dl::BM);
  const int64_t tw = tm * ceil_div(p.n, 256) * batch, tn = tm * ceil_div(p.n, 128) * batch;
  const bool w256 = dl_fits(p, b_kcont, 256) && tw < (1LL << 31) && ceil_div(p.n, 128) % 2 == 0;
  const bool w128 = dl_fits(p, b_kcont, 128) && tn < (1LL << 31);
  // 256 x 192 tiles (8 waves of 128 x 48; K-contiguous B) where they fill
  // whole rounds of the CUs and 256-wide ones do not (QKV at N = 6144:
  // 256 tiles in one round instead of 192, or 512 in two instead of 384)
  const int64_t t192 = p.n % 192 == 0 ? tm * (p.n / 192) * batch : 0;
  if (b_kcont && t192 > 0 && t192 % kNumCUs == 0 && tw % kNumCUs != 0 && dl_fits(p, b_kcont, 192) &&
      t192 < (1LL << 31)) {
    c.kind = 192;
    c.us = static_cast<double>(t192 / kNumCUs) * dl_round_us(p.k);
    return c;
  }
  // with a workspace, 256-wide tiles whose last round is split along K
  if (w256 && batch == 1 && p.part != nullptr) {
    c.split = splitk_choice(tw, p.k);
    if (c.split.splits > 1 && c.split.bytes <= p.part_bytes) {
      c.kind = 256;
      c.us = splitk_us(c.split, p.k);
      return c;
    }
    c.split = SplitPlan{};
  }
  if (w256 && (!w128 || dl_est256(tw, p.k) <= dl_est128(tn, p.k))) {
    c.kind = 256;
    c.us = dl_est256(tw, p.k);
  } else if (w128) {
    c.kind = 128;
    c.us = dl_est128(tn, p.k);
  }
  return c;
}

// K-contiguous A, whole K tiles: the direct-load kernel, 256 or 128 columns
// wide, or 256 wide with the last round split along K; K a multiple of 8: the
// ring kernel's plans.  The time models' first choice, the ring kernel only
// where it is ahead by more than the models' error (1000 x 6144 x 4096, a tie
// in the models: 62 us on split 256-wide tiles, 75 on the ring kernel).
constexpr double kRingLead = 0.9;
struct GemmRoute {
  bool ring = false;
  RingPlan rp;
  DlChoice dc;
};
inline GemmRoute gemm_route(const GemmArgs& p, int64_t batch, bool a_kcont, bool b_kcont) {
  GemmRoute r;
  // one K tile in at most a round of 64 x 64 tiles: the register-staged
  // kernel's single stage is ahead (64^3: 3.0 us against 3.3)
  if (p.k <= 64 && !(p.m % dl::BM == 0 && p.n % 128 == 0) &&
      ceil_div(p.m, 64) * ceil_div(p.n, 64) * batch <= kNumCUs) return r;
  if (a_kcont && p.k % dl::BKD == 0 && p.k > 0 && p.vec_a && p.vec_b && (b_kcont || p.nb % 8 == 0))
    r.dc = dl_choice(p, batch, b_kcont);
  if (ring_fits(p, a_kcont, b_kcont, false)) {
    r.rp = ring_plan(batch, p.m, p.n, p.k, b_kcont, false, p.part_bytes);
    r.ring = r.rp.cfg >= 0 && (r.dc.kind == 0 || r.rp.us < kRingLead * r.dc.us);
  }
  return r;
}

// Launches the direct-load kernel (and, with a split plan, the reduce).
template <typename T, int BN, bool SWIGLU = false, int WTN_ = dl::WTN>
int launch_dl(GemmArgs& p, int64_t batch, bool b_kcont, hipStream_t st,
              const SplitPlan* plan = nullptr) {
  p.tiles_m = static_cast<int>(ceil_div(p.m, dl::BM));
  p.tiles_n = static_cast<int>(ceil_div(p.n, SWIGLU ? BN / 2 : BN));
  const int64_t tiles = static_cast<int64_t>(p.tiles_m) * p.tiles_n;
  const bool split = plan != nullptr && plan->splits > 1 && batch == 1;
  p.tail_start = static_cast<int>(split ? plan->tail_start : tiles);
  p.splits = split ? plan->splits : 1;
  p.kslice = split ? plan->kslice : 0;
  const int64_t wgs = split ? plan->tail_start + (tiles - plan->tail_start) * plan->splits : tiles;
  dim3 grid(static_cast<unsigned>(wgs), static_cast<unsigned>(batch));
  constexpr int NTH = dl::Cfg<BN, WTN_>::NT;
  if (b_kcont)
    gemm_dl_kernel<T, true, BN, SWIGLU, WTN_><<<grid, dim3(NTH), 0, st>>>(p);
  else if constexpr (!SWIGLU && (BN / 8) % 16 == 0)
    gemm_dl_kernel<T, false, BN, false, WTN_><<<grid, dim3(NTH), 0, st>>>(p);
  if (split) {
    constexpr int OUTN = SWIGLU ? BN / 2 : BN;
    dim3 rg(static_cast<unsigned>(tiles - plan->tail_start), (dl::BM * OUTN) / 1024);
    gemm_splitk_reduce<T, BN, SWIGLU><<<rg, 256, 0, st>>>(p);
  }
  return check_launch("sph_gemm");
}

// Short-K problems of at least this many 128x128 tiles run the persistent
// ring kernel (two or more tiles per workgroup on 256 CUs).
constexpr int64_t kShortkRingTiles = 2 * kNumCUs;

// Short-K kernel: K of 64 or 128, whole 128x128 tiles, K-contiguous A,
// 16-byte aligned rows everywhere, plain product, 32-bit buffer offsets.
inline bool shortk_fits(const GemmArgs& p, bool a_kcont, bool b_kcont) {
  if (!(p.k == 64 || p.k == 128) || p.m % sk::BM != 0 || p.n % sk::BN != 0 || !a_kcont ||
      !p.vec_a || !p.vec_b || !p.vec_d || p.alpha != 1.f || p.c != nullptr ||
      p.epilogue != SPH_EPI_NONE)
    return false;
  if (p.m / sk::BM * (p.n / sk::BN) >= (1LL << 31)) return false;
  constexpr int64_t kLim = (1LL << 31) - 1;
  if (p.lda > kLim / 2 || p.ldb > kLim / 2) return false;
  const int64_t a_bytes = ((sk::BM - 1) * p.lda + p.k) * 2;
  const int64_t b_bytes = b_kcont ? ((sk::BN - 1) * p.ldb + p.k) * 2 : ((p.k - 1) * p.ldb + sk::BN) * 2;
  return a_bytes < kLim && b_bytes < kLim;
}

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Operands off 16-byte chunks (an odd K, rows of odd length): with a
// workspace they are copied into rows of whole chunks, zero-padded (K to a
// multiple of 64 where it is not one of 8), and the product runs on the
// kernels above.  Taken where the time models put copy and product 10 % ahead
// of the register-staged kernel: per K column of a round of its 64 x 64 tiles
// 75 ns with row-major B (its transposing loader), 14 with K-contiguous B; 48
// and 25 for 128 x 128 tiles; the copy ~3 us + its bytes at 4.5 TB/s.
// (3001 x 3003 x 3005 row-major: 329 us register-staged, 85 padded; 1501 x 999
// x 2003 191 / 28; 333 x 4099 x 4099 K-contiguous 69 / 44.)
struct PackPlan {
  bool use = false;
  bool a = false, b = false;     // operands to copy
  int64_t kp = 0, np = 0;        // padded K, padded columns of a row-major B
  int64_t a_bytes = 0, bytes = 0;
};
constexpr int64_t kPackLimit = int64_t{256} << 20;

inline GemmArgs packed_args(const GemmArgs& p, int64_t batch, bool b_kcont, const PackPlan& pp) {
  GemmArgs q = p;
  char* w = reinterpret_cast<char*>(p.part);
  q.k = pp.kp;
  if (pp.a) {
    q.a = w;
    q.lda = pp.kp;
    q.stride_a = batch == 1 || p.stride_a == 0 ? 0 : p.m * pp.kp;
    q.vec_a = 1;
  }
  if (pp.b) {
    q.b = w + pp.a_bytes;
    q.ldb = b_kcont ? pp.kp : pp.np;
    q.stride_b = batch == 1 || p.stride_b == 0 ? 0 : (b_kcont ? p.n : pp.kp) * q.ldb;
    q.vec_b = 1;
    q.nb = pp.np;
  }
  q.part_bytes = p.part_bytes > pp.bytes ? p.part_bytes - pp.bytes : 0;
  q.part = q.part_bytes > 0 ? reinterpret_cast<float*>(w + pp.bytes) : nullptr;
  return q;
}

inline PackPlan pack_plan(const GemmArgs& p, int64_t batch, bool a_kcont, bool b_kcont) {
  PackPlan pp;
  const bool k8 = p.k % 8 == 0;
  if (!a_kcont || p.k < 64 || p.part == nullptr) return pp;
  pp.a = !p.vec_a || !k8;
  pp.b = !p.vec_b || !k8 || (!b_kcont && p.nb % 8 != 0);
  if (!pp.a && !pp.b) return pp;
  pp.kp = k8 ? p.k : ceil_div(p.k, dl::BKD) * dl::BKD;
  pp.np = b_kcont ? p.n : ceil_div(p.n, 8) * 8;
  const int64_t ba = batch > 1 && p.stride_a == 0 ? 1 : batch, bb = batch > 1 && p.stride_b == 0 ? 1 : batch;
  if (p.m > kPackLimit || p.n > kPackLimit || p.k > kPackLimit || batch > 65535) return pp;
  if (static_cast<double>(ba) * p.m * pp.kp > kPackLimit || static_cast<double>(bb) * pp.np * pp.kp > kPackLimit)
    return pp;
  pp.a_bytes = pp.a ? (ba * p.m * pp.kp * 2 + 255) / 256 * 256 : 0;
  pp.bytes = pp.a_bytes + (pp.b ? (bb * pp.np * pp.kp * 2 + 255) / 256 * 256 : 0);
  if (pp.bytes > kPackLimit || pp.bytes > p.part_bytes) return pp;
  const GemmRoute r = gemm_route(packed_args(p, batch, b_kcont, pp), batch, true, b_kcont);
  const double us = 3.0 + 2.0 * static_cast<double>(pp.bytes) / 4.5e6 +
                    (r.ring ? r.rp.us : r.dc.kind != 0 ? r.dc.us : 1e30);
  const int64_t t128 = ceil_div(p.m, 128) * ceil_div(p.n, 128) * batch;
  const int64_t t64 = ceil_div(p.m, 64) * ceil_div(p.n, 64) * batch;
  const double k = static_cast<double>(p.k);
  const double staged =
      t128 >= 128 ? 5.0 + k * (b_kcont ? 0.025 : 0.048) * std::max(1.0, static_cast<double>(t128) / kNumCUs)
                  : 5.0 + k * (b_kcont ? 0.014 : 0.075) * std::max(1.0, static_cast<double>(t64) / (2 * kNumCUs));
  // (short K on many tiles: the output is the cost, the copies only add to
  // it; 8 x 1001 x 777 x 128: 14.9 us register-staged, 18.2 padded)
  pp.use = us < 0.9 * staged && (p.k >= 256 || t128 < 128);
  return pp;
}

// One thread per 8-element chunk of a padded operand; blockIdx.y: operand.
struct PackOp {
  const uint16_t* src;
  int64_t ld, stride;
  uint16_t* dst;
  int rows, cols;
  uint32_t drows, dchunks;  // padded extent (chunks of 8)
  int batches;
};
__global__ void __launch_bounds__(256) gemm_pack_kernel(PackOp o0, PackOp o1) {
  const PackOp& o = blockIdx.y == 0 ? o0 : o1;
  const uint32_t idx = blockIdx.x * 256 + threadIdx.x;  // (at most 2^24 chunks)
  if (idx >= static_cast<uint32_t>(o.batches) * o.drows * o.dchunks) return;
  const uint32_t rowi = idx / o.dchunks;
  const int c = static_cast<int>(idx - rowi * o.dchunks) * 8;
  const int b = static_cast<int>(rowi / o.drows), r = static_cast<int>(rowi - b * o.drows);
  u32x4 v = {0u, 0u, 0u, 0u};
  if (r < o.rows) {
    const uint16_t* s = o.src + b * o.stride + r * o.ld + c;
    if (c + 8 <= o.cols) {
      v = *reinterpret_cast<const u32x4_any*>(s);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (c + e < o.cols) v[e >> 1] |= static_cast<uint32_t>(s[e]) << (16 * (e & 1));
    }
  }
  *reinterpret_cast<u32x4*>(o.dst + static_cast<int64_t>(idx) * 8) = v;
}

inline void launch_pack(const GemmArgs& p, const GemmArgs& q, int64_t batch, bool b_kcont,
                        const PackPlan& pp, hipStream_t st) {
  const uint32_t kc = static_cast<uint32_t>(pp.kp / 8);
  PackOp oa{}, ob{};
  if (pp.a)
    oa = {static_cast<const uint16_t*>(p.a), p.lda, p.stride_a, static_cast<uint16_t*>(const_cast<void*>(q.a)),
          static_cast<int>(p.m), static_cast<int>(p.k), static_cast<uint32_t>(p.m), kc,
          static_cast<int>(q.stride_a == 0 ? 1 : batch)};
  if (pp.b) {
    const int rows = static_cast<int>(b_kcont ? p.n : p.k), cols = static_cast<int>(b_kcont ? p.k : p.n);
    ob = {static_cast<const uint16_t*>(p.b), p.ldb, p.stride_b, static_cast<uint16_t*>(const_cast<void*>(q.b)),
          rows, cols, static_cast<uint32_t>(b_kcont ? p.n : pp.kp),
          b_kcont ? kc : static_cast<uint32_t>(pp.np / 8),
          static_cast<int>(q.stride_b == 0 ? 1 : batch)};
  }
  if (!pp.a) oa = ob;
  const auto chunks = [](const PackOp& o) { return static_cast<int64_t>(o.batches) * o.drows * o.dchunks; };
  const int64_t most = std::max(chunks(oa), chunks(ob));
  const dim3 grid(static_cast<unsigned>(ceil_div(most, 256)), pp.a && pp.b ? 2 : 1);
  gemm_pack_kernel<<<grid, 256, 0, st>>>(oa, ob);
}

// Time of the register-staged kernel on aligned operands in the caches, K up to
// ~1500 (us; fitted with the ring kernel's hot_us): per round of 512 tiles of 128
// x 128, or of 256 x 256 tiles where those give every CU one, or one round of
// 64 x 64 tiles.  Output rows off 16 bytes cost more.
inline double staged_us(const GemmArgs& p, int64_t batch, bool b_kcont) {
  const double k = static_cast<double>(p.k) * 1e-3;
  const int64_t t256 = ceil_div(p.m, 256) * ceil_div(p.n, 256) * batch;
  const int64_t t128 = ceil_div(p.m, 128) * ceil_div(p.n, 128) * batch;
  const bool odd = p.n % 8 != 0;
  if (t256 >= kNumCUs) return static_cast<double>(ceil_div(t256, kNumCUs)) * ((odd ? 17.0 : 12.7) + 36.0 * k);
  if (t128 >= 128) {
    const double one = (b_kcont ? 6.3 + 14.6 * k : 6.7 + 19.7 * k) + (odd ? 0.5 : 0.0);
    const double two = (b_kcont ? 7.3 + 19.0 * k : 7.4 + 25.6 * k) + (odd ? 1.4 : 0.0);
    const int64_t rest = t128 % (2 * kNumCUs);
    return static_cast<double>(t128 / (2 * kNumCUs)) * two + (rest > kNumCUs ? two : rest > 0 ? one : 0.0);
  }
  if (ceil_div(p.m, 64) * ceil_div(p.n, 64) * batch <= kNumCUs) return b_kcont ? 3.6 + 7.2 * k : 4.2 + 14.4 * k;
  return b_kcont ? 4.2 + 9.6 * k : 5.2 + 16.0 * k;
}

// Short K where the ring kernel's epilogue or tiles cost more than its loads
// save; by a margin where 256 x 256 tiles fill the CUs, whose times spread most.
// Of the 1180 products of the fits, 41 take more than 5 % longer than on the
// other kernel (336 with the ring kernel for all).  fp16, ring beside
// register-staged: K-contiguous B 10 x 250 x 1024 x 32 12.3 / 7.0 us, 24 x 552 x
// 512 x 128 13.3 / 11.3, 4 x 1608 x 608 x 224 16.5 / 13.1; row-major 10 x 1571 x
// 328 x 128 13.1 / 11.2.  Past the K of both fits the ring kernel is ahead (bmm of
// 250 to 500 tiles: K 1024 even, 2048 5 % ahead).
constexpr int64_t kStagedMaxK = 1536;
inline bool staged_leads(const GemmArgs& p, int64_t batch, bool b_kcont, const GemmRoute& r) {
  if (!r.ring || r.rp.splits != 1 || p.k > kStagedMaxK) return false;
  const bool large = ceil_div(p.m, 256) * ceil_div(p.n, 256) * batch >= kNumCUs;
  return staged_us(p, batch, b_kcont) < (large ? 0.85 : 0.97) * r.rp.hot_us;
}

// 9 to 16 rows times few columns with a long K that the ring kernel does not
// split (a batch, or no workspace): its tiles leave most CUs idle and each walks
// all of K, which the small-row kernel spreads over a workgroup per two columns.
// Ring beside small-row kernel, us: columns (of the whole batch) 512 x K 1024 7.3
// / 6.6, 2048 x 1024 7.4 / 9.0; 1024 x 2048 11.6 / 8.5, 2048 x 2048 11.7 / 13.7;
// 2048 x 4096 20.7 / 17, 4096 x 4096 20.8 / 24.5; 512 x 8192 38 / 10.2, 2048 x
// 8192 38 / 28, 4096 x 8192 38 / 31.
inline bool skinny16_leads(const GemmArgs& p, int64_t batch, bool a_kcont, bool b_kcont, const GemmRoute& r) {
  return p.m <= 16 && a_kcont && b_kcont && r.ring && r.rp.splits == 1 && p.k >= 1024 &&
         p.n * batch <= std::clamp<int64_t>(p.k / 2, 1024, 4096);
}

// The kernel of a call: small row counts on the streaming kernels, short K on
// theirs, then the direct-load and ring kernels; what neither takes (A
// transposed, K or rows off 16-byte chunks) on the register-staged kernel:
// 256x256 tiles when they give at least one tile per CU, else 128x128 (more
// workgroups for the 256 CUs), else 64x64 for small problems.  With padded
// copies, the kernel is that of the product on them.
struct GemmChoice {
  sph_gemm_kernel kernel = SPH_GEMM_STAGED;
  PackPlan pack;
  RingPlan ring;
  DlChoice dl;
};
GemmChoice gemm_choice(const GemmArgs& p, int64_t batch, bool a_kcont, bool b_kcont, bool packed = false) {
  GemmChoice c;
  if (stream_fits(p, batch, a_kcont, b_kcont)) {
    c.kernel = SPH_GEMM_STREAM;
    return c;
  }
  if (p.m <= kSmallRows && a_kcont && b_kcont && p.vec_a && p.vec_b && p.k > 0 && p.k % 8 == 0 &&
      ceil_div(p.n, 2) < (1LL << 40)) {
    c.kernel = SPH_GEMM_SKINNY;
    return c;
  }
  if (shortk_fits(p, a_kcont, b_kcont)) {
    // persistent from two tiles per workgroup on: one workgroup per CU
    const int64_t tiles = p.m / sk::BM * (p.n / sk::BN) * batch;
    c.kernel = tiles >= kShortkRingTiles && p.n / sk::BN >= 2 ? SPH_GEMM_SHORT_K_RING : SPH_GEMM_SHORT_K;
    return c;
  }
  const PackPlan pp = packed ? PackPlan{} : pack_plan(p, batch, a_kcont, b_kcont);
  if (pp.use) {  // (aligned: packs nothing more)
    c = gemm_choice(packed_args(p, batch, b_kcont, pp), batch, true, b_kcont, true);
    c.pack = pp;
    return c;
  }
  const GemmRoute r = gemm_route(p, batch, a_kcont, b_kcont);
  if (skinny16_leads(p, batch, a_kcont, b_kcont, r)) {
    c.kernel = SPH_GEMM_SKINNY;
    return c;
  }
  c.ring = r.rp;
  c.dl = r.dc;
  bool ring = r.ring;
  if (!packed && staged_leads(p, batch, b_kcont, r)) {
    ring = false;
    if (p.m % dl::BM != 0 || p.n % 128 != 0) c.dl.kind = 0;  // whole tiles stay direct-load
  }
  c.kernel = ring ? SPH_GEMM_RING : c.dl.kind != 0 ? SPH_GEMM_DIRECT : SPH_GEMM_STAGED;
  return c;
}

template <typename T>
int gemm_dispatch(GemmArgs& p, int64_t batch, bool a_kcont, bool b_kcont, hipStream_t st) {
  const GemmChoice c = gemm_choice(p, batch, a_kcont, b_kcont);
  if (c.pack.use) {
    GemmArgs q = packed_args(p, batch, b_kcont, c.pack);
    launch_pack(p, q, batch, b_kcont, c.pack, st);
    p = q;
    a_kcont = true;
  }
  constexpr bool bf16 = __is_same(T, bf16_t);
  switch (c.kernel) {
    case SPH_GEMM_STREAM: return launch_stream(bf16, p, false, false, st);
    case SPH_GEMM_SKINNY: return launch_skinny(bf16, p, batch, false, st);
    case SPH_GEMM_SHORT_K_RING: {
      p.tiles_m = static_cast<int>(p.m / sk::BM);
      p.tiles_n = static_cast<int>(p.n / sk::BN);
      p.batches = batch;
      const dim3 grid(static_cast<unsigned>(kNumCUs));
      constexpr int RWM = 2, RWN = 2, RNT = skr::L<RWM, RWN>::NT;
      if (p.k == 64) {
        if (b_kcont) gemm_shortk_ring_kernel<T, true, 1, RWM, RWN><<<grid, dim3(RNT), 0, st>>>(p);
        else gemm_shortk_ring_kernel<T, false, 1, RWM, RWN><<<grid, dim3(RNT), 0, st>>>(p);
      } else {
        if (b_kcont) gemm_shortk_ring_kernel<T, true, 2, RWM, RWN><<<grid, dim3(RNT), 0, st>>>(p);
        else gemm_shortk_ring_kernel<T, false, 2, RWM, RWN><<<grid, dim3(RNT), 0, st>>>(p);
      }
      return check_launch("sph_gemm (short K)");
    }
    case SPH_GEMM_SHORT_K: {
      p.tiles_m = static_cast<int>(p.m / sk::BM);
      p.tiles_n = static_cast<int>(p.n / sk::BN);
      dim3 grid(static_cast<unsigned>(p.tiles_m) * p.tiles_n, static_cast<unsigned>(batch));
      if (p.k == 64) {
        if (b_kcont) gemm_shortk_kernel<T, true, 1><<<grid, dim3(sk::NT), 0, st>>>(p);
        else gemm_shortk_kernel<T, false, 1><<<grid, dim3(sk::NT), 0, st>>>(p);
      } else {
        if (b_kcont) gemm_shortk_kernel<T, true, 2><<<grid, dim3(sk::NT), 0, st>>>(p);
        else gemm_shortk_kernel<T, false, 2><<<grid, dim3(sk::NT), 0, st>>>(p);
      }
      return check_launch("sph_gemm (short K)");
    }
    case SPH_GEMM_RING: return launch_ring(bf16, p, batch, b_kcont, false, c.ring, st);
    case SPH_GEMM_DIRECT:
      if (c.dl.kind == 256) return launch_dl<T, 256>(p, batch, b_kcont, st, &c.dl.split);
      if (c.dl.kind == 192) return launch_dl<T, 192, false, 48>(p, batch, b_kcont, st);
      return launch_dl<T, 128, false, 32>(p, batch, b_kcont, st);
    default: return launch_staged(bf16, p, batch, a_kcont, b_kcont, st);
  }
}

}  // namespace
}  // namespace sph

using namespace sph;

namespace {
int gemm_entry(sph_dtype dtype, int trans_a, int trans_b, int64_t batch, int64_t m, int64_t n,
               int64_t k, float alpha, const void* a, int64_t lda, int64_t stride_a,
               const void* b, int64_t ldb, int64_t stride_b, float beta, const void* c,
               int64_t ldc_row, int64_t ldc_col, int64_t stride_c, void* d, int64_t ldd,
               int64_t stride_d, int epilogue, void* workspace, int64_t workspace_bytes,
               sph_stream_t stream) {
  SPH_REQUIRE(m >= 0 && n >= 0 && k >= 0 && batch >= 0, SPH_ERR_INVALID_ARG,
              "gemm: negative size");
  SPH_REQUIRE(dtype == SPH_F16 || dtype == SPH_BF16, SPH_ERR_UNSUPPORTED,
              "gemm: dtype must be F16 or BF16");
  SPH_REQUIRE(epilogue >= SPH_EPI_NONE && epilogue <= SPH_EPI_SILU,
              SPH_ERR_INVALID_ARG, "gemm: bad epilogue");
  if (m == 0 || n == 0 || batch == 0) return SPH_OK;
  SPH_REQUIRE(batch <= 65535, SPH_ERR_TOO_LARGE, "gemm: batch > 65535");
  SPH_REQUIRE(ldd >= n, SPH_ERR_INVALID_ARG, "gemm: ldd < n");
  SPH_REQUIRE(k == 0 || (trans_a ? lda >= m : lda >= k), SPH_ERR_INVALID_ARG,
              "gemm: lda too small");
  SPH_REQUIRE(k == 0 || (trans_b ? ldb >= k : ldb >= n), SPH_ERR_INVALID_ARG,
              "gemm: ldb too small");
  SPH_REQUIRE(ceil_div(m, 64) * ceil_div(n, 64) < (1LL << 31), SPH_ERR_TOO_LARGE,
              "gemm: too many tiles");
  GemmArgs p{};
  p.m = m;
  p.n = p.nb = n;
  p.k = k;
  p.a = a;
  p.lda = lda;
  p.stride_a = stride_a;
  p.b = b;
  p.ldb = ldb;
  p.stride_b = stride_b;
  p.c = (beta != 0.f) ? c : nullptr;
  p.ldc_row = ldc_row;
  p.ldc_col = ldc_col;
  p.stride_c = stride_c;
  p.d = d;
  p.ldd = ldd;
  p.stride_d = stride_d;
  p.alpha = alpha;
  p.beta = beta;
  p.epilogue = epilogue;
  // A is K-contiguous unless transposed; B is K-contiguous when transposed.
  const bool a_kcont = !trans_a, b_kcont = trans_b != 0;
  // 16-byte vector loads need aligned bases and leading dims (and batch
  // strides) that keep every row aligned.
  p.vec_a = al16(a) && (lda % 8 == 0) && (batch == 1 || stride_a % 8 == 0);
  p.vec_b = al16(b) && (ldb % 8 == 0) && (batch == 1 || stride_b % 8 == 0);
  p.vec_d = al16(d) && (ldd % 8 == 0) && (batch == 1 || stride_d % 8 == 0);
  p.part = workspace != nullptr && workspace_bytes > 0 ? static_cast<float*>(workspace) : nullptr;
  p.part_bytes = p.part != nullptr ? workspace_bytes : 0;
  hipStream_t st = as_stream(stream);
  if (dtype == SPH_F16) return gemm_dispatch<half_t>(p, batch, a_kcont, b_kcont, st);
  return gemm_dispatch<bf16_t>(p, batch, a_kcont, b_kcont, st);
}
}  // namespace

extern "C" int sph_gemm_strided_batched(
    sph_dtype dtype, int trans_a, int trans_b, int64_t batch, int64_t m,
    int64_t n, int64_t k, float alpha, const void* a, int64_t lda,
    int64_t stride_a, const void* b, int64_t ldb, int64_t stride_b, float beta,
    const void* c, int64_t ldc_row, int64_t ldc_col, int64_t stride_c, void* d,
    int64_t ldd, int64_t stride_d, int epilogue, sph_stream_t stream) {
  return gemm_entry(dtype, trans_a, trans_b, batch, m, n, k, alpha, a, lda, stride_a, b, ldb,
                    stride_b, beta, c, ldc_row, ldc_col, stride_c, d, ldd, stride_d, epilogue,
                    nullptr, 0, stream);
}

namespace {
// Workspace that a call with these operands can use: padded copies and K
// slices' partial sums.
int64_t workspace_need(int64_t batch, int64_t m, int64_t n, int64_t k, bool b_kcont, int64_t lda,
                       int64_t ldb) {
  const bool al = lda % 8 == 0 && ldb % 8 == 0 && k % 8 == 0 && (b_kcont || n % 8 == 0);
  // (host time of small calls: no copy, and K too short or rows too few to slice)
  if (al && (batch != 1 || k < 512 || (b_kcont && m <= kSmallRows))) return 0;
  GemmArgs p{};
  p.m = m;
  p.n = p.nb = n;
  p.k = k;
  p.lda = lda;
  p.ldb = ldb;
  p.stride_a = m * k;
  p.stride_b = n * k;
  p.vec_a = lda % 8 == 0;
  p.vec_b = ldb % 8 == 0;
  p.vec_d = 1;
  p.part = reinterpret_cast<float*>(uintptr_t{256});
  p.part_bytes = INT64_MAX;
  const PackPlan pp = pack_plan(p, batch, true, b_kcont);
  if (pp.use) p = packed_args(p, batch, b_kcont, pp);
  const GemmRoute r = gemm_route(p, batch, true, b_kcont);
  const int64_t split = r.ring ? r.rp.bytes : r.dc.split.splits > 1 ? r.dc.split.bytes : 0;
  return (pp.use ? pp.bytes : 0) + split;
}
}  // namespace

// (for contiguous operands, either layout of B)
extern "C" int64_t sph_gemm_workspace_bytes(int64_t batch, int64_t m, int64_t n, int64_t k) {
  if (batch <= 0 || m <= 0 || n <= 0 || k <= 0) return 0;
  return std::max(workspace_need(batch, m, n, k, true, k, k), workspace_need(batch, m, n, k, false, k, n));
}

extern "C" int64_t sph_gemm_workspace_bytes_ex(int trans_a, int trans_b, int64_t batch, int64_t m,
                                               int64_t n, int64_t k, int64_t lda, int64_t ldb) {
  if (batch <= 0 || m <= 0 || n <= 0 || k <= 0 || trans_a) return 0;
  return workspace_need(batch, m, n, k, trans_b != 0, lda, ldb);
}

extern "C" int sph_gemm_ex(sph_dtype dtype, int trans_a, int trans_b, int64_t batch, int64_t m,
                           int64_t n, int64_t k, float alpha, const void* a, int64_t lda,
                           int64_t stride_a, const void* b, int64_t ldb, int64_t stride_b,
                           float beta, const void* c, int64_t ldc_row, int64_t ldc_col,
                           int64_t stride_c, void* d, int64_t ldd, int64_t stride_d, int epilogue,
                           void* workspace, int64_t workspace_bytes, sph_stream_t stream) {
  SPH_REQUIRE(workspace_bytes >= 0, SPH_ERR_INVALID_ARG, "gemm: negative workspace size");
  return gemm_entry(dtype, trans_a, trans_b, batch, m, n, k, alpha, a, lda, stride_a, b, ldb,
                    stride_b, beta, c, ldc_row, ldc_col, stride_c, d, ldd, stride_d, epilogue,
                    workspace, workspace_bytes, stream);
}

extern "C" int sph_gemm(sph_dtype dtype, int trans_a, int trans_b, int64_t m,
                        int64_t n, int64_t k, float alpha, const void* a,
                        int64_t lda, const void* b, int64_t ldb, float beta,
                        const void* c, int64_t ldc_row, int64_t ldc_col,
                        void* d, int64_t ldd, int epilogue,
                        sph_stream_t stream) {
  return sph_gemm_strided_batched(dtype, trans_a, trans_b, 1, m, n, k, alpha, a,
                                  lda, 0, b, ldb, 0, beta, c, ldc_row, ldc_col,
                                  0, d, ldd, 0, epilogue, stream);
}

namespace {
// SwiGLU route of m > 8 rows: 256-row tiles of the direct-load kernel (n %
// 128, k % 64; its last round split along K) or the ring kernel (k % 8).
struct SwigluRoute {
  bool dl = false, ring = false;
  SplitPlan split;
  RingPlan rp;
};
SwigluRoute swiglu_route(const GemmArgs& p, int64_t ws_bytes) {
  SwigluRoute r;
  constexpr int64_t kLim = 1LL << 31;
  const int64_t tiles = ceil_div(p.m, dl::BM) * (p.n / 128);
  double us = 0;
  if (p.n % 128 == 0 && p.k > 0 && p.k % dl::BKD == 0 && ((dl::BM - 1) * p.lda + p.k) * 2 < kLim &&
      ((p.n + 127) * p.ldb + p.k) * 2 < kLim && tiles < kLim) {
    r.dl = true;
    us = dl_est256(tiles, p.k);
    r.split = splitk_plan(tiles, p.k / dl::BKD, 256);
    if (r.split.splits > 1 && r.split.bytes <= ws_bytes)
      us = splitk_us(r.split, p.k);
    else
      r.split = SplitPlan{};
  }
  if (ring_fits(p, true, true, true)) {
    r.rp = ring_plan(1, p.m, p.n, p.k, true, true, ws_bytes);
    r.ring = r.rp.cfg >= 0 && (!r.dl || r.rp.us < kRingLead * us);
  }
  return r;
}

int swiglu_run(sph_dtype dtype, int64_t m, int64_t n, int64_t k, const void* a, int64_t lda,
               const void* w, int64_t ldw, void* d, int64_t ldd, void* workspace,
               int64_t workspace_bytes, hipStream_t st) {
  GemmArgs p{};
  p.m = m;
  p.n = n;
  p.k = k;
  p.a = a;
  p.lda = lda;
  p.b = w;
  p.ldb = ldw;
  p.d = d;
  p.ldd = ldd;
  p.alpha = 1.f;
  p.epilogue = SPH_EPI_NONE;
  p.vec_a = p.vec_b = 1;
  p.vec_d = al16(d) && ldd % 8 == 0;
  const SwigluRoute r = swiglu_route(p, workspace != nullptr ? workspace_bytes : 0);
  SPH_REQUIRE(r.ring || r.dl, SPH_ERR_TOO_LARGE,
              "gemm_swiglu: operands too large for 32-bit tile offsets");
  p.part = static_cast<float*>(workspace);
  if (r.ring) return launch_ring(dtype == SPH_BF16, p, 1, true, true, r.rp, st);
  if (dtype == SPH_F16) return launch_dl<half_t, 256, true>(p, 1, true, st, &r.split);
  return launch_dl<bf16_t, 256, true>(p, 1, true, st, &r.split);
}

int swiglu_stream(sph_dtype dtype, int64_t m, int64_t n, int64_t k, const void* a, int64_t lda,
                  const void* w, int64_t ldw, void* d, int64_t ldd, hipStream_t st) {
  // decode shapes: the weight-stream kernel, gate and up rows per wave
  SPH_REQUIRE(k >= 64 && k % 8 == 0 && k <= 8192 && n < (1LL << 40), SPH_ERR_UNSUPPORTED,
              "gemm_swiglu: small m needs 64 <= k <= 8192, k % 8 == 0");
  GemmArgs q{};
  q.m = m;
  q.n = n;
  q.k = k;
  q.a = a;
  q.lda = lda;
  q.b = w;
  q.ldb = ldw;
  q.d = d;
  q.ldd = ldd;
  q.alpha = 1.f;
  return launch_stream(dtype == SPH_BF16, q, true, false, st);
}

int swiglu_check(sph_dtype dtype, int64_t m, int64_t n, int64_t k, const void* a, int64_t lda,
                 const void* w, int64_t ldw, int64_t ldd) {
  SPH_REQUIRE(m >= 0 && n >= 0 && k >= 0, SPH_ERR_INVALID_ARG, "gemm_swiglu: negative size");
  SPH_REQUIRE(dtype == SPH_F16 || dtype == SPH_BF16, SPH_ERR_UNSUPPORTED,
              "gemm_swiglu: dtype must be F16 or BF16");
  if (m == 0 || n == 0) return SPH_OK;
  SPH_REQUIRE(lda >= k && ldw >= k && ldd >= n, SPH_ERR_INVALID_ARG,
              "gemm_swiglu: leading dimension too small");
  SPH_REQUIRE(al16(a) && al16(w) && lda % 8 == 0 && ldw % 8 == 0, SPH_ERR_UNSUPPORTED,
              "gemm_swiglu: rows of x and w must be 16-byte aligned");
  return SPH_OK;
}
}  // namespace

extern "C" int64_t sph_gemm_swiglu_workspace_bytes(int64_t m, int64_t n, int64_t k) {
  if (m <= 8 || n <= 0 || k <= 0 || k % 8 != 0) return 0;
  GemmArgs p{};
  p.m = m;
  p.n = n;
  p.k = p.lda = p.ldb = k;
  p.vec_a = p.vec_b = 1;
  const SwigluRoute r = swiglu_route(p, INT64_MAX);
  return r.ring ? r.rp.bytes : r.split.bytes;
}

extern "C" int sph_gemm_swiglu(sph_dtype dtype, int64_t m, int64_t n, int64_t k, const void* a,
                               int64_t lda, const void* w, int64_t ldw, void* d, int64_t ldd,
                               void* workspace, int64_t workspace_bytes, sph_stream_t stream) {
  const int rc = swiglu_check(dtype, m, n, k, a, lda, w, ldw, ldd);
  if (rc != SPH_OK || m == 0 || n == 0) return rc;
  hipStream_t st = as_stream(stream);
  if (m <= 8) return swiglu_stream(dtype, m, n, k, a, lda, w, ldw, d, ldd, st);
  SPH_REQUIRE(m % dl::BM == 0 && n % 128 == 0 && k > 0 && k % dl::BKD == 0, SPH_ERR_UNSUPPORTED,
              "gemm_swiglu: needs m <= 8, or m % 256 == 0, n % 128 == 0, k % 64 == 0");
  SPH_REQUIRE(al16(d) && ldd % 8 == 0, SPH_ERR_UNSUPPORTED,
              "gemm_swiglu: rows of d must be 16-byte aligned");
  return swiglu_run(dtype, m, n, k, a, lda, w, ldw, d, ldd, workspace, workspace_bytes, st);
}

extern "C" int sph_gemm_swiglu_any(sph_dtype dtype, int64_t m, int64_t n, int64_t k, const void* a,
                                   int64_t lda, const void* w, int64_t ldw, void* d, int64_t ldd,
                                   void* workspace, int64_t workspace_bytes, sph_stream_t stream) {
  const int rc = swiglu_check(dtype, m, n, k, a, lda, w, ldw, ldd);
  if (rc != SPH_OK || m == 0 || n == 0) return rc;
  hipStream_t st = as_stream(stream);
  if (m <= 8 && k >= 64 && k % 8 == 0 && k <= 8192)
    return swiglu_stream(dtype, m, n, k, a, lda, w, ldw, d, ldd, st);
  SPH_REQUIRE(k > 0 && k % 8 == 0, SPH_ERR_UNSUPPORTED, "gemm_swiglu: k must be a multiple of 8");
  return swiglu_run(dtype, m, n, k, a, lda, w, ldw, d, ldd, workspace, workspace_bytes, st);
}

extern "C" int sph_gemm_plan(int trans_a, int trans_b, int64_t batch, int64_t m, int64_t n,
                             int64_t k, int64_t lda, int64_t ldb, int plain, int swiglu,
                             int64_t workspace_bytes, int32_t* plan) {
  SPH_REQUIRE(plan != nullptr && batch > 0 && m > 0 && n > 0 && k > 0 && workspace_bytes >= 0,
              SPH_ERR_INVALID_ARG, "gemm_plan: sizes must be positive");
  GemmArgs p{};
  p.m = m;
  p.n = p.nb = n;
  p.k = k;
  p.lda = lda;
  p.ldb = ldb;
  p.ldd = n;
  p.stride_a = trans_a ? k * lda : m * lda;
  p.stride_b = trans_b ? n * ldb : k * ldb;
  p.vec_a = lda % 8 == 0 && (batch == 1 || p.stride_a % 8 == 0);
  p.vec_b = ldb % 8 == 0 && (batch == 1 || p.stride_b % 8 == 0);
  p.vec_d = n % 8 == 0;
  p.alpha = plain ? 1.f : 0.5f;
  p.part = workspace_bytes > 0 ? reinterpret_cast<float*>(uintptr_t{256}) : nullptr;  // (not read)
  p.part_bytes = workspace_bytes;
  GemmChoice c;
  if (swiglu) {
    SPH_REQUIRE(!trans_a && trans_b && batch == 1 && k % 8 == 0 && p.vec_a && p.vec_b,
                SPH_ERR_UNSUPPORTED, "gemm_plan: not a SwiGLU product");
    if (m <= 8 && k >= 64 && k <= 8192) {
      c.kernel = SPH_GEMM_STREAM;
    } else {
      const SwigluRoute r = swiglu_route(p, workspace_bytes);
      SPH_REQUIRE(r.ring || r.dl, SPH_ERR_TOO_LARGE, "gemm_plan: operands too large");
      c.kernel = r.ring ? SPH_GEMM_RING : SPH_GEMM_DIRECT;
      c.ring = r.rp;
      c.dl.kind = 256;
      c.dl.split = r.split;
    }
  } else {
    c = gemm_choice(p, batch, !trans_a, trans_b != 0);
  }
  const bool ring = c.kernel == SPH_GEMM_RING, dl_ = c.kernel == SPH_GEMM_DIRECT;
  plan[0] = c.kernel;
  plan[1] = ring ? c.ring.bm : dl_ ? static_cast<int>(dl::BM) : 0;
  plan[2] = ring ? c.ring.bn : dl_ ? c.dl.kind : 0;
  plan[3] = ring ? c.ring.splits : dl_ ? c.dl.split.splits : 1;
  plan[4] = (c.pack.a ? 1 : 0) + (c.pack.b ? 2 : 0);
  plan[5] = ring ? c.ring.cfg : -1;
  return SPH_OK;
}

extern "C" int sph_gemm_rmsnorm(sph_dtype dtype, int64_t m, int64_t n, int64_t k, const void* a,
                                int64_t lda, const void* norm_w, float eps, const void* w,
                                int64_t ldw, void* d, int64_t ldd, int swiglu,
                                sph_stream_t stream) {
  SPH_REQUIRE(dtype == SPH_F16 || dtype == SPH_BF16, SPH_ERR_UNSUPPORTED,
              "gemm_rmsnorm: dtype must be F16 or BF16");
  SPH_REQUIRE(m >= 0 && n >= 0 && k >= 0, SPH_ERR_INVALID_ARG, "gemm_rmsnorm: negative size");
  if (m == 0 || n == 0) return SPH_OK;
  SPH_REQUIRE(m <= 8, SPH_ERR_UNSUPPORTED, "gemm_rmsnorm: at most 8 rows (decode shapes)");
  SPH_REQUIRE(k >= 64 && k % 8 == 0 && k <= 8192, SPH_ERR_UNSUPPORTED,
              "gemm_rmsnorm: needs 64 <= k <= 8192, k % 8 == 0");
  SPH_REQUIRE(std::isfinite(eps) && eps >= 0.f, SPH_ERR_INVALID_ARG,
              "gemm_rmsnorm: eps must be finite and >= 0");
  SPH_REQUIRE(lda >= k && ldw >= k && ldd >= n && n < (1LL << 40), SPH_ERR_INVALID_ARG,
              "gemm_rmsnorm: leading dimension too small");
  SPH_REQUIRE(al16(a) && al16(w) && al16(norm_w) && lda % 8 == 0 && ldw % 8 == 0,
              SPH_ERR_UNSUPPORTED, "gemm_rmsnorm: x, norm_w and w rows must be 16-byte aligned");
  GemmArgs q{};
  q.m = m;
  q.n = n;
  q.k = k;
  q.a = a;
  q.lda = lda;
  q.b = w;
  q.ldb = ldw;
  q.d = d;
  q.ldd = ldd;
  q.alpha = 1.f;
  q.epilogue = SPH_EPI_NONE;
  q.vec_a = q.vec_b = 1;
  q.vec_d = al16(d) && ldd % 8 == 0;
  q.norm_w = norm_w;
  q.norm_eps = eps;
  hipStream_t st = as_stream(stream);
  const bool bf16 = dtype == SPH_BF16;
  // (swiglu: w holds the gate rows [0, n) and the up rows [n, 2n))
  if (swiglu || stream_fits(q, 1, true, true)) return launch_stream(bf16, q, swiglu != 0, true, st);
  return launch_skinny(bf16, q, 1, true, st);
}

extern "C" int sph_gemm_f16(int64_t m, int64_t n, int64_t k, const void* a,
                            const void* b, void* d, sph_stream_t stream) {
  return sph_gemm(SPH_F16, 0, 0, m, n, k, 1.0f, a, k, b, n, 0.0f, nullptr, 0, 0,
                  d, n, SPH_EPI_NONE, stream);
}

extern "C" int sph_bmm_f16(int64_t batch, int64_t m, int64_t n, int64_t k,
                           const void* a, const void* b, void* d,
                           sph_stream_t stream) {
  return sph_gemm_strided_batched(SPH_F16, 0, 0, batch, m, n, k, 1.0f, a, k,
                                  m * k, b, n, k * n, 0.0f, nullptr, 0, 0, 0, d,
                                  n, m * n, SPH_EPI_NONE, stream);
}
