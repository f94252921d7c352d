// Products whose rows do not fill the 256-row tiles of the direct-load
// kernel: decode batches above 8, short prompts, ragged row counts.
//
//   * Tiles of 32 x 64 to 192 x 128 on 4 waves (2 x 2), two or three
//     workgroups per CU, or 128 x 128 on 8.  At small M the cost is reading B
//     (a weight matrix) once, so the kernel is built around keeping B bytes
//     in flight: ST - 1 K tiles of a ring of ST LDS stages are loading while
//     one is multiplied (48-80 KB of LDS per workgroup, 128-160 KB per CU).
//   * Operands move global -> LDS by buffer_load_dwordx4 ... lds from raw
//     buffer resources that end at the operand's last row: rows past M or N
//     read zeros, so ragged tiles need no bounds checks.  In a last, partial
//     K tile the lanes whose 16-byte chunk lies past K take an offset outside
//     the resource and fill their LDS slot with zeros.
//   * The K range is split over workgroups until the chip is full (fp32
//     partial sums in a caller's workspace, added in a fixed order by
//     gemm_ring_reduce, which applies the epilogue).  Arrival counters
//     instead of the second launch would need device-scope releases, each an
//     L2 write-back on this 8-XCD part.
//   * The MFMAs take B as the first operand: a lane then holds 4 consecutive
//     output columns of one row.  K slices store those as they lie; unsplit
//     products pass 16 rows at a time through LDS, so that stores cover whole
//     tile rows.
#include <algorithm>

#include "gemm_ring.h"

namespace sph {
namespace {

template <typename T>
__device__ inline u32x2 pack4(f32x4 v) {
  u32x2 w;
#pragma unroll
  for (int e = 0; e < 2; ++e)
    w[e] = static_cast<uint32_t>(__builtin_bit_cast(uint16_t, Num<T>::from_f(v[2 * e]))) |
           (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, Num<T>::from_f(v[2 * e + 1]))) << 16);
  return w;
}

// Four output columns of one row: epilogue (unless done: SwiGLU) and store.
template <typename T, bool PLAIN>
__device__ inline void store4(const GemmArgs& p, T* D, f32x4 v, int64_t bz, int row, int col) {
  if constexpr (!PLAIN) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < p.n) v[e] = epilogue_one<T>(p, v[e], bz, row, col + e);
  }
  T* dp = D + row * p.ldd + col;
  if (col + 4 <= p.n) {
    typedef u32x2 u32x2_any __attribute__((aligned(2)));
    *reinterpret_cast<u32x2_any*>(dp) = pack4<T>(v);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < p.n) dp[e] = Num<T>::from_f(v[e]);
  }
}

namespace ring {
constexpr uint32_t kOutside = 0x80000000u;  // past every buffer resource

// Tile BM x BN on NW waves (2 x NW / 2), K tiles of BK, ST ring stages.
template <int BM_, int BN_, int NW_, int BK_, int ST_>
struct Cfg {
  static constexpr int BM = BM_, BN = BN_, NW = NW_, BK = BK_, ST = ST_, NT = NW * 64;
  static constexpr int CPR = BK / 8, KK = BK / 32;  // 16-byte chunks, MFMA sub-steps per K tile
  static constexpr int WM = 2, WN = NW / 2, WTM = BM / WM, WTN = BN / WN;
  static constexpr int TM = WTM / 16, TN = WTN / 16;
  static constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2, STAGE = A_BYTES + B_BYTES;
  static constexpr int LA = A_BYTES / 1024 / NW, LB = B_BYTES / 1024 / NW, L = LA + LB;
  static constexpr int BCH = BN / 8;  // 16-byte chunks per row-major B row
  static_assert(LA * NW * 1024 == A_BYTES && LB * NW * 1024 == B_BYTES, "DMA lines");
  static_assert(WTM % 16 == 0 && WTN % 16 == 0, "wave tile");
  static_assert((ST - 2) * L < 64, "vmcnt range");
  static_assert(BK == 32 || BK == 64, "swizzle");
  // Chunk c of K-contiguous row r sits at slot c ^ swz(r): the 16 rows that a
  // fragment read touches at one chunk then cover all 64 banks.
  __device__ static inline int swz(int r) { return BK == 64 ? (r >> 1) & 7 : (r >> 2) & 3; }
};
}  // namespace ring

// Waits until at most `tiles` K tiles of L loads each are still in flight.
template <int ST, int L>
__device__ inline void wait_tiles(int tiles) {
  static_assert(ST <= 4, "at most two tiles in flight behind the one awaited");
  if constexpr (ST >= 4) {
    if (tiles >= 2) return wait_vmcnt<2 * L>();
  }
  if constexpr (ST >= 3) {
    if (tiles >= 1) return wait_vmcnt<L>();
  }
  wait_vmcnt<0>();
}

// SWIGLU: B holds the gate rows [0, n) and the up rows [n, 2n) of one weight
// matrix; a tile covers BN / 2 output columns, 16 gate rows and the 16 up
// rows of the same columns alternating, so a wave's MFMA columns 2j and
// 2j + 1 hold the two sums of the same outputs.
template <typename T, bool B_KCONT, bool SWIGLU, int BM_, int BN_, int NW_, int BK_, int ST_>
__global__ void __launch_bounds__(NW_ * 64) gemm_ring_kernel(const GemmArgs p) {
  using C = ring::Cfg<BM_, BN_, NW_, BK_, ST_>;
  constexpr int BK = C::BK, CPR = C::CPR, KK = C::KK;
  constexpr int BM = C::BM, BN = C::BN, TM = C::TM, TN = C::TN, ST = C::ST, L = C::L;
  constexpr int OUTN = SWIGLU ? BN / 2 : BN;
  static_assert(B_KCONT || C::BCH % 16 == 0, "row-major B: the swizzle needs 16-chunk rows");
  static_assert(!SWIGLU || (B_KCONT && TN % 2 == 0), "gate / up column pairs");
  __shared__ __attribute__((aligned(1024))) char lds[ST * C::STAGE];

  // Workgroup -> (tile, K slice).  Dispatch is round-robin over 8 XCDs: give
  // each XCD a contiguous run, row tiles of one B panel next to each other.
  int id = blockIdx.x;
  {
    const int total = gridDim.x, q = total >> 3, r = total & 7, x = id & 7;
    id = x * q + min(x, r) + (id >> 3);
  }
  const int tm = id % p.tiles_m;
  id /= p.tiles_m;
  const int split = id % p.splits, tn = id / p.splits;
  const int64_t bz = blockIdx.y;
  const int m0 = tm * BM, n0 = tn * OUTN;
  const int m = static_cast<int>(p.m), n = static_cast<int>(p.n), k = static_cast<int>(p.k);
  const int lda = static_cast<int>(p.lda), ldb = static_cast<int>(p.ldb);
  const int kt_all = (k + BK - 1) / BK;
  const int kt0 = split * p.kslice;
  const int ksteps = min(p.kslice, kt_all - kt0);
  const uint16_t* A = static_cast<const uint16_t*>(p.a) + bz * p.stride_a + static_cast<int64_t>(m0) * lda;
  const uint16_t* B = static_cast<const uint16_t*>(p.b) + bz * p.stride_b +
                      (B_KCONT ? static_cast<int64_t>(n0) * ldb : n0);
  const int arows = min(BM, m - m0);
  const int brows = SWIGLU    ? 2 * n - n0
                    : B_KCONT ? min(BN, n - n0)
                              : min(BN, static_cast<int>(p.nb) - n0);  // columns
  const i32x4 ra = buffer_rsrc(A, static_cast<uint32_t>((arows - 1) * lda + k) * 2u);
  const i32x4 rb = buffer_rsrc(B, B_KCONT ? static_cast<uint32_t>((brows - 1) * ldb + k) * 2u
                                          : static_cast<uint32_t>((k - 1) * ldb + brows) * 2u);

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / C::WN, wn = wave % C::WN;
  uint32_t va[C::LA], vb[C::LB];
#pragma unroll
  for (int i = 0; i < C::LA; ++i) {
    const int s = (wave * C::LA + i) * 64 + lane;
    const int r = s / CPR, c = (s % CPR) ^ C::swz(r);
    // rows past M: outside the resource (r * lda may wrap back into it)
    va[i] = r < arows ? static_cast<uint32_t>(r * lda * 2 + c * 16) : ring::kOutside;
  }
#pragma unroll
  for (int i = 0; i < C::LB; ++i) {
    const int s = (wave * C::LB + i) * 64 + lane;
    if constexpr (B_KCONT) {
      const int r = s / CPR, c = (s % CPR) ^ C::swz(r);
      const int wr = SWIGLU ? 16 * (r >> 5) + (r & 15) + ((r & 16) ? n : 0) : r;
      vb[i] = wr < brows ? static_cast<uint32_t>(wr * ldb * 2 + c * 16) : ring::kOutside;
    } else {
      const int kr = s / C::BCH, c = (s % C::BCH) ^ bswz(kr);
      vb[i] = c * 8 < brows ? static_cast<uint32_t>(kr * ldb * 2 + c * 16) : ring::kOutside;
    }
  }
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((SPH_LDS char*)(lds)));

  // DMA of K tile t (of this slice) into ring slot `slot`.
  auto issue = [&](int t, int slot) __attribute__((always_inline)) {
    const int kt = kt0 + t;
    const uint32_t sbase = lds_base + slot * C::STAGE;
    const int kleft = k - kt * BK;  // < BK: partial last K tile
    const uint32_t sa = kt * BK * 2, sb = B_KCONT ? sa : static_cast<uint32_t>(kt * BK * ldb * 2);
#pragma unroll
    for (int i = 0; i < C::LA; ++i) {
      uint32_t v = va[i];
      if (kleft < BK) {
        const int s = (wave * C::LA + i) * 64 + lane;
        const int c = (s % CPR) ^ C::swz(s / CPR);
        if (c * 8 >= kleft) v = ring::kOutside;
      }
      dma16(ra, __builtin_amdgcn_readfirstlane(sbase + (wave * C::LA + i) * 1024), v,
            __builtin_amdgcn_readfirstlane(sa));
    }
#pragma unroll
    for (int i = 0; i < C::LB; ++i) {
      uint32_t v = vb[i];
      if (kleft < BK) {
        const int s = (wave * C::LB + i) * 64 + lane;
        if constexpr (B_KCONT) {
          const int c = (s % CPR) ^ C::swz(s / CPR);
          if (c * 8 >= kleft) v = ring::kOutside;
        } else {
          if (s / C::BCH >= kleft) v = ring::kOutside;
        }
      }
      dma16(rb, __builtin_amdgcn_readfirstlane(sbase + C::A_BYTES + (wave * C::LB + i) * 1024), v,
            __builtin_amdgcn_readfirstlane(sb));
    }
  };

  // Fragment reads: as in the direct-load kernel.
  const int m16 = lane & 15, g4 = lane >> 4, sw = g4 ^ C::swz(m16);
  int aoff[KK], bkoff[KK], boff[TN];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
    aoff[kk] = (wm * C::WTM + m16) * (CPR * 16) + ((sw ^ (4 * kk)) << 4);
    bkoff[kk] = C::A_BYTES + (wn * C::WTN + m16) * (CPR * 16) + ((sw ^ (4 * kk)) << 4);
  }
  if constexpr (!B_KCONT) {
    const int e = m16 >> 2, q = m16 & 3;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int nn = wn * C::WTN + j * 16 + 4 * q;
      boff[j] = C::A_BYTES + (8 * g4 + e) * (BN * 2) + (((nn >> 3) ^ bswz(8 * g4 + e)) << 4) + 8 * (q & 1);
    }
  }

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int t = 0; t < ST - 1 && t < ksteps; ++t) issue(t, t);
  int slot = 0;
  for (int ks = 0; ks < ksteps; ++ks) {
    // tile ks has landed once only the later tiles' loads are outstanding;
    // the barrier also means every wave is done with the slot of tile ks - 1
    wait_tiles<ST, L>(min(ST - 2, ksteps - 1 - ks));
    wait_lgkmcnt0();
    __syncthreads();
    if (ks + ST - 1 < ksteps) issue(ks + ST - 1, slot == 0 ? ST - 1 : slot - 1);
    const char* sp = lds + slot * C::STAGE;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      u32x4 af[TM], bf[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (B_KCONT) {
          bf[j] = *reinterpret_cast<const u32x4*>(sp + bkoff[kk] + j * 16 * CPR * 16);
        } else {
          u32x2 h[2];
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) {
            const SPH_LDS char* bp = (const SPH_LDS char*)(sp) + boff[j] + (kk * 32 + 4 * hh) * (BN * 2);
            h[hh] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((SPH_LDS s16x4*)(bp)));
          }
          bf[j] = __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3);
        }
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = *reinterpret_cast<const u32x4*>(sp + aoff[kk] + i * 16 * CPR * 16);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mfma16<T>(bf[j], af[i], acc[i][j]);
    }
    slot = slot + 1 == ST ? 0 : slot + 1;
  }

  // Lane: row l % 16 of MFMA tile i, columns 4 (l / 16) .. + 3 of tile j.
  const int row0 = m0 + wm * C::WTM + m16;
  if (p.splits > 1) {
    const int np = (n + 3) & ~3;  // partial rows: np columns (SwiGLU: gate, then up)
    const int64_t pitch = SWIGLU ? 2 * np : np;
    float* W = p.part + static_cast<int64_t>(split) * m * pitch;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = row0 + 16 * i;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int col = n0 + (SWIGLU ? wn * (C::WTN / 2) + 16 * (j >> 1) : wn * C::WTN + 16 * j) + 4 * g4;
        if (row < m && col < np)
          *reinterpret_cast<f32x4*>(W + row * pitch + (SWIGLU && (j & 1) ? np : 0) + col) = acc[i][j];
      }
    }
    return;
  }
  // Each wave stages 16 rows of its tile in LDS (its own part of the ring:
  // every DMA has landed, the barrier ends the other waves' reads) and stores
  // them 16 bytes a lane, whole tile rows at a time: 8-byte stores of the
  // accumulators as they lie write 32-byte pieces (8 x 3108 x 777 x 128: 49.4
  // us, 37.6 through LDS).
  T* D = static_cast<T*>(p.d) + bz * p.stride_d;
  constexpr int TO = SWIGLU ? TN / 2 : TN, WO = TO * 16;  // output columns of the wave
  constexpr int CPO = WO / 8, RPI = 64 / CPO;             // 16-byte chunks per row, rows per store
  constexpr int SP = WO + 8;                               // slab pitch (elements)
  static_assert(C::NW * 16 * SP * 2 <= ST * C::STAGE, "slabs fit the ring");
  __syncthreads();
  T* slab = reinterpret_cast<T*>(lds) + wave * (16 * SP);
  const int colw = n0 + wn * WO;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = row0 + 16 * i;
#pragma unroll
    for (int j = 0; j < TO; ++j) {
      const int col = colw + 16 * j + 4 * g4;
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (SWIGLU)
          v[e] = silu(acc[i][2 * j][e]) * acc[i][2 * j + 1][e];
        else
          v[e] = row < m && col + e < n ? epilogue_one<T>(p, acc[i][j][e], bz, row, col + e) : 0.f;
      }
      *reinterpret_cast<u32x2*>(slab + m16 * SP + 16 * j + 4 * g4) = pack4<T>(v);
    }
    wait_lgkmcnt0();
#pragma unroll
    for (int r = 0; r < 16; r += RPI) {
      const int rr = r + lane / CPO, cc = (lane % CPO) * 8;
      const int orow = m0 + wm * C::WTM + 16 * i + rr, ocol = colw + cc;
      if (rr < 16 && orow < m && ocol < n) {
        const u32x4 w = *reinterpret_cast<const u32x4*>(slab + rr * SP + cc);
        T* dp = D + orow * p.ldd + ocol;
        if (ocol + 8 <= n) {
          *reinterpret_cast<u32x4_any*>(dp) = w;
        } else {
          const T* e = reinterpret_cast<const T*>(&w);
#pragma unroll
          for (int q = 0; q < 8; ++q)
            if (ocol + q < n) dp[q] = e[q];
        }
      }
    }
    wait_lgkmcnt0();
  }
}

// Adds the K slices' sums in slice order and applies the epilogue: one
// thread per 4 output columns of a row (16-byte reads of every slice).
template <typename T, bool SWIGLU>
__global__ void __launch_bounds__(256) gemm_ring_reduce(const GemmArgs p) {
  const int m = static_cast<int>(p.m), n = static_cast<int>(p.n), nq = (n + 3) >> 2;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= m * nq) return;
  const int row = idx / nq, col = (idx - row * nq) * 4;
  const int64_t pitch = SWIGLU ? 8 * nq : 4 * nq, step = m * pitch;
  const float* W = p.part + row * pitch + col;
  f32x4 v = {0.f, 0.f, 0.f, 0.f}, u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < p.splits; ++s) {
    v += *reinterpret_cast<const f32x4*>(W + s * step);
    if constexpr (SWIGLU) u += *reinterpret_cast<const f32x4*>(W + s * step + 4 * nq);
  }
  if constexpr (SWIGLU) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = silu(v[e]) * u[e];
  }
  store4<T, SWIGLU>(p, static_cast<T*>(p.d), v, 0, row, col);
}

template <typename T, bool B_KCONT, bool SWIGLU, int BM, int BN, int NW, int BK, int ST>
void launch(GemmArgs& p, int64_t batch, hipStream_t st) {
  p.tiles_m = static_cast<int>(ceil_div(p.m, BM));
  p.tiles_n = static_cast<int>(ceil_div(p.n, SWIGLU ? BN / 2 : BN));
  const dim3 grid(static_cast<unsigned>(p.tiles_m) * p.tiles_n * p.splits, static_cast<unsigned>(batch));
  gemm_ring_kernel<T, B_KCONT, SWIGLU, BM, BN, NW, BK, ST><<<grid, dim3(NW * 64), 0, st>>>(p);
  if (p.splits > 1) {
    const int64_t quads = p.m * ceil_div(p.n, 4);
    gemm_ring_reduce<T, SWIGLU><<<static_cast<unsigned>(ceil_div(quads, 256)), 256, 0, st>>>(p);
  }
}

// Tile configurations.  per_cu workgroups share a CU (LDS); ns[w - 1] is the
// time per K column, in ns, of a workgroup when w of them do, `bk` its K
// tile.  Measured on one MI355X with weights from HBM (fp16, us):
//   32 x 64    24 x 6144 x 4096 in 5 slices 15.0, 24 x 4096 x 4096 in 4 11.5
//   64 x 128   64 x 6144 x 4096 in 5 slices 17.1, 333 x 6144 x 4096 39.4
//   128 x 128 on 8 waves   128 x 6144 x 4096 in 4 slices 21.8, 777 x 4096 x 4096 42.9
//   128 x 128 on 4 waves   333 x 6144 x 4096 in 3 slices 36.6, 333 x 4096 x 12800 in 5 59.5
//   192 x 128  2331 x 4096 x 4096 102.6, 333 x 2*12800 x 4096 (SwiGLU) 111.7
// (the kernels these products ran on before: 24 rows 60-140 us, 333 x 6144 x
// 4096 64 us).  Not kept, from the same sweep of 16 products (us
// beside the best tile above): 128 x 128 with 3 to 5 stages of 32-deep K tiles
// (41.7 beside 36.6 at 333 x 6144 x 4096, 170.4 beside 144.9 at 2331 x 6144 x
// 4096; within 4 % at 128 x 6144); 128 x 256 tiles (107.8 beside 102.6 at
// 2331 x 4096 x 4096, nowhere the fastest); 96-row tiles (nowhere among the
// first seven).  256-row tiles were 2-3 % faster on two (142.3 beside 144.9 at
// 2331 x 6144, which gemm.hip's 256-row tiles take, and 28.7 beside 29.6 at
// 200 x 6144) and slower on the others: not worth an instance.
struct RingCfg {
  int bm, bn, bk, per_cu;
  double ns[3];
  bool kcont_only;
};
constexpr RingCfg kRing[] = {
    {32, 64, 64, 3, {3.2, 6.6, 9.0}, true},  {32, 128, 64, 2, {6.0, 9.0, 0}, false},
    {64, 128, 64, 2, {8.0, 12.0, 0}, false}, {128, 128, 64, 1, {9.3, 0, 0}, false},
    {128, 128, 64, 2, {11.0, 16.5, 0}, false}, {192, 128, 32, 2, {16.0, 25.0, 0}, true}};
constexpr int kRingCfgs = sizeof(kRing) / sizeof(kRing[0]);
constexpr int64_t kCUs = 256;

// Unsplit products of K up to ~1500 with operands in the caches: us per round of
// workgroups, fixed and per 1000 K columns, with one, two or three workgroups
// on the CUs, in the order of kRing (128 x 128 tiles on 4 waves, third: one on
// the CUs behind a full round).  Fitted to 1180 products (both layouts of B,
// 40 to 3000 rows and 40 to 6000 columns in batches of 1 to 64, K 8 to 3072).
// What the plan's model leaves out is the second workgroup's epilogue (128 x
// 128 tiles, 480 of them, K 32: 11.5 us against 7.0 for 160 at K 64) and the 192
// x 128 tile's (160, K 32: 12.3 us).
constexpr double kHot[kRingCfgs][3][2] = {
    {{1.5, 4.0}, {1.6, 6.0}, {2.2, 8.0}}, {{2.4, 5.5}, {3.0, 9.0}, {}},
    {{4.0, 7.6}, {4.3, 12.0}, {}},        {{4.3, 10.8}, {}, {}},
    {{4.2, 11.0}, {8.5, 17.2}, {8.3, 11.0}}, {{12.5, 18.5}, {12.5, 34.3}, {}}};
double hot_us(int cfg, int64_t wgs, int64_t k) {
  const int64_t slots = kCUs * kRing[cfg].per_cu, rest = wgs % slots;
  const double kk = static_cast<double>(k) * 1e-3;
  auto round = [&](int64_t load) { return kHot[cfg][load][0] + kHot[cfg][load][1] * kk; };
  double us = 2.0 + static_cast<double>(wgs / slots) * round(kRing[cfg].per_cu - 1);
  const bool behind = wgs > slots && rest <= kCUs && kHot[cfg][2][0] > 0.0 && kRing[cfg].per_cu == 2;
  if (rest > 0) us += round(behind ? 2 : (rest - 1) / kCUs);
  return us;
}

}  // namespace

// Time of a plan: ~2 us of launch and, per round of workgroups, ~4 us of first
// bytes and output plus the K columns of the fullest CU, but no less than the
// operands' time from HBM (~5.2 TB/s); a K split adds the reduce launch (~2 us) and its partial sums'
// write and read (~6 TB/s, mostly from the caches).  At least 256 K columns
// a slice and at most 8 slices: past that the partial sums cost more than
// the shorter slices save (24 x 4096 x 4096: 4 slices 11.5 us, 8 12.4).
RingPlan ring_plan(int64_t batch, int64_t m, int64_t n, int64_t k, bool b_kcont, bool swiglu,
                   int64_t max_bytes) {
  RingPlan best;
  const int64_t nw = swiglu ? 2 * n : n;
  const double mem_us = 2.0 * batch * (m * k + nw * k + m * n) / 5.2e6 + 5.0;
  for (int c = 0; c < kRingCfgs; ++c) {
    const RingCfg& f = kRing[c];
    if (f.kcont_only && !b_kcont) continue;
    const int64_t tiles = batch * ceil_div(m, f.bm) * ceil_div(nw, f.bn);
    const int64_t ktiles = ceil_div(k, f.bk);
    for (int s = 1; s <= 8; ++s) {
      if (s > 1 && (batch != 1 || tiles * s > 2 * kCUs * f.per_cu || k < 256 * s)) break;
      const int64_t slice = ceil_div(ktiles, s);
      if (s > 1 && ceil_div(ktiles, slice) != s) continue;  // every slice non-empty
      const int64_t bytes = s > 1 ? s * m * ((n + 3) / 4 * 4) * (swiglu ? 8 : 4) : 0;
      if (bytes > max_bytes || bytes >= (int64_t{1} << 31)) continue;
      const int64_t wgs = tiles * s, slots = kCUs * f.per_cu, rest = wgs % slots;
      double ns = static_cast<double>(wgs / slots) * f.ns[f.per_cu - 1];
      if (rest > 0) ns += f.ns[(rest - 1) / kCUs];
      double us = 2.0 + 4.0 * static_cast<double>(ceil_div(wgs, slots)) +
                  static_cast<double>(slice * f.bk) * ns * 1e-3;
      us = us > mem_us ? us : mem_us;
      if (s > 1) us += 2.0 + 2.0 * static_cast<double>(bytes) / 6e6;
      if (best.cfg < 0 || us < best.us) {
        best.cfg = c;
        best.bm = f.bm;
        best.bn = f.bn;
        best.splits = s;
        best.kslice = static_cast<int>(slice);
        best.bytes = bytes;
        best.us = us;
        best.hot_us = s == 1 ? hot_us(c, wgs, k) : 0;
      }
    }
  }
  return best;
}

bool ring_fits(const GemmArgs& p, bool a_kcont, bool b_kcont, bool swiglu) {
  constexpr int64_t kLim = (int64_t{1} << 31) - 1;
  if (!a_kcont || !p.vec_a || !p.vec_b || p.k <= 0 || p.k % 8 != 0) return false;
  if (!b_kcont && p.nb % 8 != 0) return false;
  if (p.m >= kLim / 4 || p.n >= kLim / 4 || p.k >= kLim / 4) return false;
  if (p.lda > kLim / 4 || p.ldb > kLim / 4) return false;
  const int64_t brows = swiglu ? 2 * p.n : 128;
  const int64_t a_bytes = (191 * p.lda + p.k) * 2;
  const int64_t b_bytes = b_kcont ? (brows * p.ldb + p.k) * 2 : (p.k * p.ldb + 128) * 2;
  // (the K tile past the last one is never addressed; 64 columns of slack)
  if (a_bytes >= kLim || b_bytes + 64 * (b_kcont ? 2 : 2 * p.ldb) >= kLim) return false;
  return ceil_div(p.m, 32) * ceil_div(p.n, 32) * 8 < kLim && p.m * ceil_div(p.n, 4) < kLim;
}

namespace {
template <typename T, bool B_KCONT, bool SWIGLU>
void launch_cfg(GemmArgs& p, int64_t batch, int cfg, hipStream_t st) {
  switch (cfg) {
    case 0:
      if constexpr (B_KCONT) launch<T, true, SWIGLU, 32, 64, 4, 64, 4>(p, batch, st);
      break;
    case 1: launch<T, B_KCONT, SWIGLU, 32, 128, 4, 64, 4>(p, batch, st); break;
    case 2: launch<T, B_KCONT, SWIGLU, 64, 128, 4, 64, 3>(p, batch, st); break;
    case 3: launch<T, B_KCONT, SWIGLU, 128, 128, 8, 64, 4>(p, batch, st); break;
    case 4: launch<T, B_KCONT, SWIGLU, 128, 128, 4, 64, 2>(p, batch, st); break;
    default:
      if constexpr (B_KCONT) launch<T, true, SWIGLU, 192, 128, 4, 32, 3>(p, batch, st);
  }
}
template <typename T>
void launch_t(GemmArgs& p, int64_t batch, bool b_kcont, bool swiglu, int cfg, hipStream_t st) {
  if (swiglu)
    launch_cfg<T, true, true>(p, batch, cfg, st);
  else if (b_kcont)
    launch_cfg<T, true, false>(p, batch, cfg, st);
  else
    launch_cfg<T, false, false>(p, batch, cfg, st);
}
}  // namespace

int launch_ring(bool bf16, GemmArgs& p, int64_t batch, bool b_kcont, bool swiglu,
                const RingPlan& plan, hipStream_t st) {
  p.splits = plan.splits;
  p.kslice = plan.kslice;
  if (bf16)
    launch_t<bf16_t>(p, batch, b_kcont, swiglu, plan.cfg, st);
  else
    launch_t<half_t>(p, batch, b_kcont, swiglu, plan.cfg, st);
  return check_launch("sph_gemm (ring)");
}

}  // namespace sph
