// Products with at most 8 rows of A whose operands are both K-contiguous
// (decode steps and LM heads: x[M, K] times an nn.Linear weight W[N, K]): they
// are HBM-bound on reading W once and run as streams of packed dot products,
// which keep every CU on its own rows of W, with an RMSNorm prologue and a
// SwiGLU epilogue.  (From 9 rows on the MFMA ring kernel is ahead: 16 x 6144 x
// 4096 32.9 us here, 16.8 there; 8 x 6144 x 4096 17.2 here.  Up to 16 rows run
// here where that kernel cannot split a long K over the CUs and has few tiles.)
#include <algorithm>

#include "gemm_route.h"

namespace sph {
namespace {

// x * w elementwise on 8 packed 2-byte values, each product rounded to T;
// adds the squares of x's values to ss.
template <typename T>
__device__ inline u32x4 norm_chunk(u32x4 x, u32x4 w, float& ss) {
  const T* xe = reinterpret_cast<const T*>(&x);
  const T* we = reinterpret_cast<const T*>(&w);
  u32x4 r;
  T* re = reinterpret_cast<T*>(&r);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float xf = Num<T>::to_f(xe[e]);
    ss = fmaf(xf, xf, ss);
    re[e] = Num<T>::from_f(xf * Num<T>::to_f(we[e]));
  }
  return r;
}


// ---------------------------------------------------------------------------
// Small-M products: D[m, n] = epi(alpha * sum_k A[m, k] * B[n, k] + beta*C)
// for M <= MT rows, A and B K-contiguous and 16-byte aligned, K % 8 == 0.
// A group of TPR threads computes R output columns n for all M rows: thread t
// reads 16 bytes of each of the R weight rows at k = 8t + 8*TPR*j (whole row
// segments per group, coalesced) and keeps the R loads of two K steps in
// flight.  TPR follows K (256 threads for K >= 2048 down to 16 for K = 128,
// so short rows such as attention keys do not idle most of the workgroup)
// and a workgroup holds 256/TPR groups.  Workgroups loop over row blocks
// (grid capped near the number of resident workgroups), so long matrices do
// not end in a partial wave of workgroups.  A (at most 16 x K, read by every
// workgroup) comes through the caches.  fp16 uses v_dot2_f32_f16, bf16
// v_dot2_f32_bf16 (two products summed into an fp32 accumulator; subnormals
// kept).  With bf16 widened into fp32 FMAs the vector ALUs set the time: 4 x
// 6144 x 4096 15.3 us against 13.0, 8 x 49155 x 4096 112 against 83, gate / up of
// 8 x 12800 x 4096 59.7 against 47.3, the same error against 64 bits.  Partial
// sums are reduced within the group by butterflies and, for groups wider than a
// wave, through LDS.
// ---------------------------------------------------------------------------
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

template <typename T>
__device__ inline float dot8_acc(u32x4 a, u32x4 b, float acc) {
  if constexpr (__is_same(T, half_t)) {
    // (vector elements are copied to scalars first: this compiler lowers
    // __builtin_bit_cast of an indexed vector element to element 0)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t ai = a[i], bi = b[i];
      acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, ai), __builtin_bit_cast(f16x2, bi),
                                   acc, false);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t ai = a[i], bi = b[i];
      acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, ai), __builtin_bit_cast(bf16x2, bi),
                                            acc, false);
    }
  }
  return acc;
}

constexpr int kSkinnyThreads = 256;

// NORM: the RMSNorm prologue of GemmArgs (norm_w, norm_eps) on A's rows.
template <typename T, int MT, int R, int TPR, bool NORM = false>
__global__ void __launch_bounds__(kSkinnyThreads) gemm_skinny_kernel(const GemmArgs p,
                                                                     int64_t nblocks) {
  constexpr int G = kSkinnyThreads / TPR;   // row groups per workgroup
  constexpr int WPG = TPR > 64 ? TPR / 64 : 1;  // waves per group
  __shared__ float red[TPR > 64 ? G * WPG * MT * R : 1];
  __shared__ float red_ss[NORM && TPR > 64 ? G * WPG * MT : 1];
  const int g = threadIdx.x / TPR, t = threadIdx.x % TPR;
  const int64_t bz = blockIdx.y;
  const uint16_t* A = static_cast<const uint16_t*>(p.a) + bz * p.stride_a;
  const uint16_t* B = static_cast<const uint16_t*>(p.b) + bz * p.stride_b;
  const uint16_t* NW = static_cast<const uint16_t*>(p.norm_w);
  T* D = static_cast<T*>(p.d) + bz * p.stride_d;
  const int mrows = static_cast<int>(p.m);
  const float inv_k = 1.0f / static_cast<float>(p.k);
  // Every thread runs the same number of outer iterations (the bound does
  // not depend on the group), so the barriers below are uniform.
  for (int64_t base = static_cast<int64_t>(blockIdx.x) * G; base < nblocks;
       base += static_cast<int64_t>(gridDim.x) * G) {
    const int64_t blk = base + g;
    const int64_t n0 = blk * R;
    float acc[MT][R];
    float ss[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      ss[m] = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) acc[m][r] = 0.f;
    }
    if (blk < nblocks) {
      // Loads are unconditional (rows past N and M read a valid row, whose
      // results are never stored) so no branch separates them: the R + MT
      // loads of the next K step are issued before the current step's dot
      // products and one wait covers them.
      const uint16_t* bp[R];
#pragma unroll
      for (int r = 0; r < R; ++r) bp[r] = B + (n0 + r < p.n ? n0 + r : p.n - 1) * p.ldb;
      const uint16_t* ap[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) ap[m] = A + (m < mrows ? m : mrows - 1) * p.lda;
      constexpr int64_t STEP = TPR * 8;
      int64_t k = static_cast<int64_t>(t) * 8;
      if (k < p.k) {
        u32x4 w[R], x[MT], nw = zero4();
#pragma unroll
        for (int r = 0; r < R; ++r)
          w[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(bp[r] + k));
#pragma unroll
        for (int m = 0; m < MT; ++m) x[m] = *reinterpret_cast<const u32x4*>(ap[m] + k);
        if constexpr (NORM) nw = *reinterpret_cast<const u32x4*>(NW + k);
        while (true) {
          const int64_t kn = k + STEP;
          const bool more = kn < p.k;
          const int64_t kl = more ? kn : k;  // reload the current step when done
          u32x4 w2[R], x2[MT], nw2 = zero4();
#pragma unroll
          for (int r = 0; r < R; ++r)
            w2[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(bp[r] + kl));
#pragma unroll
          for (int m = 0; m < MT; ++m) x2[m] = *reinterpret_cast<const u32x4*>(ap[m] + kl);
          if constexpr (NORM) nw2 = *reinterpret_cast<const u32x4*>(NW + kl);
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const u32x4 xm = NORM ? norm_chunk<T>(x[m], nw, ss[m]) : x[m];
#pragma unroll
            for (int r = 0; r < R; ++r) acc[m][r] = dot8_acc<T>(xm, w[r], acc[m][r]);
          }
          if (!more) break;
#pragma unroll
          for (int r = 0; r < R; ++r) w[r] = w2[r];
#pragma unroll
          for (int m = 0; m < MT; ++m) x[m] = x2[m];
          nw = nw2;
          k = kn;
        }
      }
    }
    // Butterflies within the group's wave segment (all lanes take part).
    constexpr int LANES = TPR > 64 ? 64 : TPR;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int off = LANES / 2; off > 0; off >>= 1)
          acc[m][r] += __shfl_xor(acc[m][r], off, 64);
      if constexpr (NORM) {
#pragma unroll
        for (int off = LANES / 2; off > 0; off >>= 1) ss[m] += __shfl_xor(ss[m], off, 64);
      }
    }
    if constexpr (TPR > 64) {
      const int wig = t / 64;  // wave within the group
      if ((t & 63) == 0) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
          for (int r = 0; r < R; ++r) red[((g * WPG) + wig) * MT * R + m * R + r] = acc[m][r];
          if constexpr (NORM) red_ss[((g * WPG) + wig) * MT + m] = ss[m];
        }
      }
      __syncthreads();
      for (int q = t; q < MT * R; q += TPR) {
        const int m = q / R, r = q % R;
        const int64_t n = n0 + r;
        if (blk < nblocks && m < mrows && n < p.n) {
          float v = 0.f, sq = 0.f;
#pragma unroll
          for (int w = 0; w < WPG; ++w) {
            v += red[(g * WPG + w) * MT * R + q];
            if constexpr (NORM) sq += red_ss[(g * WPG + w) * MT + m];
          }
          if constexpr (NORM) v *= rsqrtf(sq * inv_k + p.norm_eps);
          D[m * p.ldd + n] = Num<T>::from_f(epilogue_one<T>(p, v, bz, m, n));
        }
      }
      __syncthreads();
    } else {
      if (blk < nblocks) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const int64_t n = n0 + r;
            if (t == (m * R + r) % TPR && m < mrows && n < p.n) {
              float v = acc[m][r];
              if constexpr (NORM) v *= rsqrtf(ss[m] * inv_k + p.norm_eps);
              D[m * p.ldd + n] = Num<T>::from_f(epilogue_one<T>(p, v, bz, m, n));
            }
          }
      }
    }
  }
}

template <typename T, int MT, int R, int TPR, bool NORM = false>
void launch_skinny_cfg(const GemmArgs& p, int64_t batch, hipStream_t st) {
  const int64_t nblocks = ceil_div(p.n, R);
  constexpr int G = kSkinnyThreads / TPR;
  int64_t gx = ceil_div(nblocks, G);
  const int64_t cap = batch >= 4096 ? 1 : 4096 / batch;
  if (gx > cap) gx = cap;
  dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(batch));
  gemm_skinny_kernel<T, MT, R, TPR, NORM><<<grid, dim3(kSkinnyThreads), 0, st>>>(p, nblocks);
}

// Launch shape from a sweep on MI355X over the decode shapes (x[4, K] times
// W[N, K], 32 MB .. 400 MB of weights): two-wave groups (TPR 128) with two
// columns each for K ~ 4096, four columns for long rows, one-wave groups of
// four columns for very wide W (LM heads), whole-workgroup groups for narrow
// W; TPR never exceeds K / 8 (every thread owns at least one K chunk).
template <typename T, int MT, bool NORM = false>
void launch_skinny_m(const GemmArgs& p, int64_t batch, hipStream_t st) {
  int tmax = 256;
  while (tmax > 16 && static_cast<int64_t>(tmax) * 8 > p.k) tmax >>= 1;
  const int64_t cols = p.n * batch;
  int tpr = 128, r = p.k >= 8192 ? 4 : 2;
  if (cols >= 32768) tpr = 64, r = 4;
  else if (cols <= 2048) tpr = 256, r = 2;
  if (tpr > tmax) tpr = tmax, r = 2;
  if (r == 4 && tpr == 64) return launch_skinny_cfg<T, MT, 4, 64, NORM>(p, batch, st);
  if (r == 4) return launch_skinny_cfg<T, MT, 4, 128, NORM>(p, batch, st);
  switch (tpr) {
    case 256: return launch_skinny_cfg<T, MT, 2, 256, NORM>(p, batch, st);
    case 128: return launch_skinny_cfg<T, MT, 2, 128, NORM>(p, batch, st);
    case 64: return launch_skinny_cfg<T, MT, 2, 64, NORM>(p, batch, st);
    case 32: return launch_skinny_cfg<T, MT, 2, 32, NORM>(p, batch, st);
    default: return launch_skinny_cfg<T, MT, 2, 16, NORM>(p, batch, st);
  }
}

template <typename T, bool NORM>
void skinny_t(const GemmArgs& p, int64_t batch, hipStream_t st) {
  if (p.m <= 1)
    launch_skinny_m<T, 1, NORM>(p, batch, st);
  else if (p.m <= 4)
    launch_skinny_m<T, 4, NORM>(p, batch, st);
  else if (NORM || p.m <= 8)
    launch_skinny_m<T, 8, NORM>(p, batch, st);
  else if constexpr (!NORM) {  // (skinny16_leads: few columns, long rows)
    if (p.n * batch > 2048)  // (K >= 4096: 8 x 10 x 512 x 8192 31 us, 42 in two columns)
      launch_skinny_cfg<T, 16, 4, 128>(p, batch, st);
    else if (p.k >= 2048)
      launch_skinny_cfg<T, 16, 2, 256>(p, batch, st);
    else
      launch_skinny_cfg<T, 16, 2, 128>(p, batch, st);
  }
}

// ---------------------------------------------------------------------------
// Decode-shaped products (M <= 8 activation rows against a weight matrix
// W[N, K] read once; batch 1, K from 1024 to 16384): the weight stream is
// the whole cost, so the kernel is built to keep as many weight bytes in
// flight as the CU allows and to give every wave the same share of them.
//   * One workgroup of WV waves per CU (persistent over the rows; 16 waves,
//     or 12 / 10 where that makes the rows whole rounds of the grid): the
//     M x K activations are staged into LDS once and read from there
//     (16-byte chunks, a wave's 64 lanes on 1 KB of consecutive bytes).
//   * Each wave streams whole weight rows: lane l owns the 16-byte chunks
//     l, l + 64, ... of the row, in segments of SEG chunks.  The wave walks
//     a flat sequence of (row, segment) items and loads item i+1 into one
//     register buffer while it computes item i from the other, so loads of
//     the next row are in flight while a row's sums are reduced and stored.
//   * Rows go round-robin over all W waves of the grid for the N / W whole
//     rounds.  The N % W rows left over would leave most waves idle for a
//     whole row time (gate/up of a 4096-wide model: 12800 rows = 3.125
//     rounds of 4096), so each of them is split along K between Q waves of
//     one workgroup (Q = 16 / the workgroup's leftover rows, rounded to a
//     power of two): the slice is the last item of each of those waves, and
//     after one workgroup barrier the first wave of each group adds the Q
//     partial sums from LDS and writes the outputs.
//   * At the end of a row the 64 lane sums per activation row are reduced by
//     butterflies and one lane writes the M outputs (with the epilogue:
//     alpha, beta*C, activation).
// ---------------------------------------------------------------------------
namespace gv {
constexpr int WAVES = 16, SEG = 8;
}

// SWIGLU: W holds the gate rows [0, n) and the up rows [n, 2n); output j
// is silu(x W[j]) * (x W[n + j]).  A wave's item then loads SEG / 2 chunks
// of both rows (the same register footprint) and the end of the row
// combines the two sums.
// NORM: the RMSNorm prologue of GemmArgs (norm_w, norm_eps), applied while
// the activations are staged (sums of squares reduced through LDS at the
// staging barrier) and to the finished sums of each row.
template <typename T, int MT, int KMAX, bool SWIGLU = false, bool NORM = false,
          int WV = gv::WAVES>
__global__ void __launch_bounds__(WV * 64) gemm_stream_kernel(const GemmArgs p) {
  using gv::SEG;
  constexpr int WAVES = WV, THREADS = WV * 64;
  constexpr int NR = SWIGLU ? 2 : 1, SEGK = SEG / NR;  // rows per item, chunks per row
  __shared__ __attribute__((aligned(16))) uint16_t As[MT * KMAX];
  __shared__ float lds_ss[NORM ? WAVES * MT : 1];
  __shared__ float lds_part[WAVES * NR * MT];  // partial sums of split rows
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nc = static_cast<int>(p.k / 8);           // 16-byte chunks per row
  const int mrows = static_cast<int>(p.m);
  const uint16_t* A = static_cast<const uint16_t*>(p.a);
  const uint16_t* B = static_cast<const uint16_t*>(p.b);
  T* D = static_cast<T*>(p.d);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * WAVES;  // W
  const int64_t rounds = p.n / stride;                 // whole rounds
  const int64_t main_end = rounds * stride;            // rows [0, main_end) whole
  const int64_t left = p.n - main_end;                 // rows split along K
  // This wave's slice of a split row: group `slot` of `qn` waves shares
  // leftover row main_end + slot * gridDim.x + blockIdx.x; this wave holds
  // chunks [tcb, tcb + tcn) of it.
  int qn = 1, q = 0, slot = 0, tcb = 0, tcn = 0;
  int64_t trow = -1;
  if (left > 0) {
    const int64_t G = gridDim.x;
    const int rpw = static_cast<int>((left + G - 1) / G);  // <= WAVES
    int p2 = 1;
    while (p2 < rpw) p2 <<= 1;
    qn = WAVES / p2;
    while (qn > 1 && nc / qn < 64) qn >>= 1;  // at least one chunk per lane
    slot = wave / qn;
    q = wave % qn;
    const int64_t t = static_cast<int64_t>(slot) * G + blockIdx.x;
    if (slot < rpw && t < left) {
      trow = main_end + t;
      const int cs = (nc + qn - 1) / qn;
      tcb = q * cs;
      tcn = nc - tcb < cs ? nc - tcb : cs;
    }
  }
  const int nseg = ((nc + 63) / 64 + SEGK - 1) / SEGK;            // segments of a row
  const int tseg = ((tcn + 63) / 64 + SEGK - 1) / SEGK;           // of this wave's slice
  u32x4 wa[SEG], wb[SEG];
  float acc[NR][MT];
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[r][m] = 0.f;

// Weight chunks of item (ROW_, chunks from CB_, segment SEG_) into register
// buffer W_ (row r of the item in entries r * SEGK ..; chunks past the
// range read a valid chunk that is not summed).
#define SPH_GV_LOAD(W_, ROW_, CB_, SEG_)                                                    \
  do {                                                                                      \
    _Pragma("unroll") for (int r_ = 0; r_ < NR; ++r_) {                                     \
      const uint16_t* rp_ = B + ((ROW_) + r_ * p.n) * p.ldb;                                \
      _Pragma("unroll") for (int j_ = 0; j_ < SEGK; ++j_) {                                 \
        int c_ = (CB_) + ((SEG_) * SEGK + j_) * 64 + lane;                                  \
        c_ = c_ < nc ? c_ : nc - 1;                                                         \
        W_[r_ * SEGK + j_] =                                                                \
            __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(rp_ + c_ * 8));       \
      }                                                                                     \
    }                                                                                       \
  } while (0)
#define SPH_GV_COMPUTE(W_, CB_, CE_, SEG_)                                                  \
  do {                                                                                      \
    _Pragma("unroll") for (int j_ = 0; j_ < SEGK; ++j_) {                                   \
      const int c_ = (CB_) + ((SEG_) * SEGK + j_) * 64 + lane;                              \
      if (c_ < (CE_)) {                                                                     \
        _Pragma("unroll") for (int m_ = 0; m_ < MT; ++m_) {                                 \
          const u32x4 a_ = *reinterpret_cast<const u32x4*>(As + (m_ * nc + c_) * 8);        \
          _Pragma("unroll") for (int r_ = 0; r_ < NR; ++r_)                                 \
              acc[r_][m_] = dot8_acc<T>(a_, W_[r_ * SEGK + j_], acc[r_][m_]);               \
        }                                                                                   \
      }                                                                                     \
    }                                                                                       \
  } while (0)
#define SPH_GV_REDUCE()                                                                     \
  _Pragma("unroll") for (int r_ = 0; r_ < NR; ++r_)                                         \
    _Pragma("unroll") for (int m_ = 0; m_ < MT; ++m_)                                       \
      _Pragma("unroll") for (int o_ = 32; o_ > 0; o_ >>= 1)                                 \
          acc[r_][m_] += __shfl_xor(acc[r_][m_], o_, 64)
// Output of row ROW_ from its two (SWIGLU) or one sums S0_(m), S1_(m):
// lane m < M writes element (m, ROW_).
#define SPH_GV_STORE(ROW_, S0_, S1_)                                                        \
  do {                                                                                      \
    float v_ = 0.f;                                                                         \
    _Pragma("unroll") for (int m_ = 0; m_ < MT; ++m_) {                                     \
      const float g_ = (S0_) * rs[m_];                                                      \
      const float x_ = SWIGLU ? silu(g_) * ((S1_) * rs[m_]) : g_;                           \
      v_ = lane == m_ ? x_ : v_;                                                            \
    }                                                                                       \
    if (lane < MT && lane < mrows)                                                          \
      D[lane * p.ldd + (ROW_)] = Num<T>::from_f(                                            \
          SWIGLU ? v_ : epilogue_one<T>(p, v_, 0, lane, (ROW_)));                        \
  } while (0)
// End of item (ROW_, SEG_) when it completes a row or a slice.
#define SPH_GV_FINISH(ROW_, TAIL_)                                                          \
  do {                                                                                      \
    SPH_GV_REDUCE();                                                                        \
    if (TAIL_) {                                                                            \
      if (lane == 0) {                                                                      \
        _Pragma("unroll") for (int r_ = 0; r_ < NR; ++r_)                                   \
          _Pragma("unroll") for (int m_ = 0; m_ < MT; ++m_)                                 \
            lds_part[(wave * NR + r_) * MT + m_] = acc[r_][m_];                             \
      }                                                                                     \
    } else {                                                                                \
      SPH_GV_STORE(ROW_, acc[0][m_], acc[NR - 1][m_]);                                      \
    }                                                                                       \
    _Pragma("unroll") for (int r_ = 0; r_ < NR; ++r_)                                       \
      _Pragma("unroll") for (int m_ = 0; m_ < MT; ++m_) acc[r_][m_] = 0.f;                  \
  } while (0)

  // This wave's item sequence: segments 0..nseg-1 of rows n0, n0 + W, ...
  // below main_end, then segments 0..tseg-1 of its split-row slice.
  int64_t n = static_cast<int64_t>(blockIdx.x) * WAVES + wave;
  int cb = 0, ce = nc, ns = nseg, s = 0;
  bool tail = false, have = n < main_end;
  if (!have && trow >= 0) {
    n = trow, cb = tcb, ce = tcb + tcn, ns = tseg, tail = true, have = true;
  }
  // The first weight loads go out before the activations are staged, so
  // the two latencies overlap.
  if (have) SPH_GV_LOAD(wa, n, cb, 0);
  // Stage the activations ([m][chunk], rows past M as zeros).
  float rs[MT];  // row scales of the RMSNorm prologue (1 without it)
#pragma unroll
  for (int m = 0; m < MT; ++m) rs[m] = 0.f;
  for (int i = threadIdx.x; i < MT * nc; i += THREADS) {
    const int m = i / nc, c = i - m * nc;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (m < mrows) v = *reinterpret_cast<const u32x4*>(A + m * p.lda + c * 8);
    if constexpr (NORM) {
      float sq = 0.f;
      v = norm_chunk<T>(v, *reinterpret_cast<const u32x4*>(
                               static_cast<const uint16_t*>(p.norm_w) + c * 8), sq);
#pragma unroll
      for (int mm = 0; mm < MT; ++mm) rs[mm] += mm == m ? sq : 0.f;
    }
    *reinterpret_cast<u32x4*>(As + (m * nc + c) * 8) = v;
  }
  if constexpr (NORM) {
#pragma unroll
    for (int mm = 0; mm < MT; ++mm) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) rs[mm] += __shfl_xor(rs[mm], o, 64);
      if (lane == 0) lds_ss[wave * MT + mm] = rs[mm];
    }
  }
  __syncthreads();
  if constexpr (NORM) {
    const float inv_k = 1.0f / static_cast<float>(p.k);
#pragma unroll
    for (int mm = 0; mm < MT; ++mm) {
      float sq = 0.f;
      for (int w = 0; w < WAVES; ++w) sq += lds_ss[w * MT + mm];
      rs[mm] = rsqrtf(sq * inv_k + p.norm_eps);
    }
  } else {
#pragma unroll
    for (int m = 0; m < MT; ++m) rs[m] = 1.f;
  }
  // Items in order; item i+1 loads while item i computes.  (The next item
  // of the last segment of a row: the next whole row, else the slice.)
#define SPH_GV_NEXT(N2_, CB2_, CE2_, NS2_, S2_, T2_, MORE_)                                  \
  do {                                                                                      \
    N2_ = n, CB2_ = cb, CE2_ = ce, NS2_ = ns, S2_ = s + 1, T2_ = tail, MORE_ = true;        \
    if (S2_ == ns) {                                                                        \
      S2_ = 0;                                                                              \
      if (!tail && n + stride < main_end) {                                                 \
        N2_ = n + stride;                                                                   \
      } else if (!tail && trow >= 0) {                                                      \
        N2_ = trow, CB2_ = tcb, CE2_ = tcb + tcn, NS2_ = tseg, T2_ = true;                  \
      } else {                                                                              \
        MORE_ = false;                                                                      \
      }                                                                                     \
    }                                                                                       \
  } while (0)
  if (have) {
    while (true) {
      int64_t n2;
      int cb2, ce2, ns2, s2;
      bool t2, more;
      SPH_GV_NEXT(n2, cb2, ce2, ns2, s2, t2, more);
      if (more) SPH_GV_LOAD(wb, n2, cb2, s2);
      SPH_GV_COMPUTE(wa, cb, ce, s);
      if (s == ns - 1) SPH_GV_FINISH(n, tail);
      if (!more) break;
      n = n2, cb = cb2, ce = ce2, ns = ns2, s = s2, tail = t2;
      SPH_GV_NEXT(n2, cb2, ce2, ns2, s2, t2, more);
      if (more) SPH_GV_LOAD(wa, n2, cb2, s2);
      SPH_GV_COMPUTE(wb, cb, ce, s);
      if (s == ns - 1) SPH_GV_FINISH(n, tail);
      if (!more) break;
      n = n2, cb = cb2, ce = ce2, ns = ns2, s = s2, tail = t2;
    }
  }
  if (left > 0) {
    // uniform: `left` is the same for every wave of the grid
    __syncthreads();
    if (trow >= 0 && q == 0) {
      float s0[MT], s1[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) s0[m] = s1[m] = 0.f;
      for (int qq = 0; qq < qn; ++qq) {
        const int w = slot * qn + qq;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          s0[m] += lds_part[(w * NR) * MT + m];
          s1[m] += lds_part[(w * NR + NR - 1) * MT + m];
        }
      }
      SPH_GV_STORE(trow, s0[m_], s1[m_]);
    }
  }
#undef SPH_GV_NEXT
#undef SPH_GV_LOAD
#undef SPH_GV_COMPUTE
#undef SPH_GV_REDUCE
#undef SPH_GV_STORE
#undef SPH_GV_FINISH
}

// Waves per workgroup: 16, or 12 / 10 where that makes the N rows whole
// rounds of the 256-workgroup grid, so that no row is left to split along K
// (decode QKV: 6144 rows = 2 rounds of 12 waves, 15.7 -> 14.0 us; gate/up:
// 12800 rows = 5 rounds of 10 waves, 41.5 -> 39.0 us; measured on MI355X).
constexpr int64_t kStreamCUs = 256;  // one workgroup per MI355X compute unit
inline int stream_waves(int64_t n) {
  if (n % (kStreamCUs * gv::WAVES) == 0) return gv::WAVES;
  for (int w : {12, 10})
    if (n % (kStreamCUs * w) == 0) return w;
  return gv::WAVES;
}

template <typename T, int MT, int KMAX, bool SWIGLU, bool NORM>
void launch_stream_k(const GemmArgs& p, hipStream_t st) {
  const int w = stream_waves(p.n);
  const int64_t wgs = ceil_div(p.n, static_cast<int64_t>(w));
  const unsigned grid = static_cast<unsigned>(wgs < kStreamCUs ? wgs : kStreamCUs);
  if (w == 12)
    gemm_stream_kernel<T, MT, KMAX, SWIGLU, NORM, 12><<<grid, dim3(12 * 64), 0, st>>>(p);
  else if (w == 10)
    gemm_stream_kernel<T, MT, KMAX, SWIGLU, NORM, 10><<<grid, dim3(10 * 64), 0, st>>>(p);
  else
    gemm_stream_kernel<T, MT, KMAX, SWIGLU, NORM, 16><<<grid, dim3(16 * 64), 0, st>>>(p);
}

template <typename T, bool SWIGLU, bool NORM>
void launch_stream_t(const GemmArgs& p, hipStream_t st) {
  if (p.m > 4)
    launch_stream_k<T, 8, 8192, SWIGLU, NORM>(p, st);
  else if (!SWIGLU && !NORM && p.k > 8192)
    launch_stream_k<T, 4, 16384, false, false>(p, st);
  else
    launch_stream_k<T, 4, 8192, SWIGLU, NORM>(p, st);
}
template <typename T>
void launch_stream_d(const GemmArgs& p, bool swiglu, bool norm, hipStream_t st) {
  if (swiglu && norm)
    launch_stream_t<T, true, true>(p, st);
  else if (swiglu)
    launch_stream_t<T, true, false>(p, st);
  else if (norm)
    launch_stream_t<T, false, true>(p, st);
  else
    launch_stream_t<T, false, false>(p, st);
}

}  // namespace

// Streaming kernel fit: batch 1, M <= 8, K-contiguous 16-byte aligned rows,
// K % 8 == 0 within the LDS staging size (16384 for M <= 4, else 8192),
// and at least 8 M weights (16 MB of fp16): with the leftover rows split
// along K every wave streams the same share, which beats the small-M
// kernel's many short workgroups from the decode step's 32 MB O projection
// up (measured on MI355X, x[4, 4096] and x[4, 12800]).
constexpr int64_t kStreamMinWeights = 8LL << 20;

bool stream_fits(const GemmArgs& p, int64_t batch, bool a_kcont, bool b_kcont) {
  return batch == 1 && p.m >= 1 && p.m <= 8 && a_kcont && b_kcont && p.vec_a && p.vec_b &&
         p.k >= 1024 && p.k % 8 == 0 && p.k <= (p.m <= 4 ? 16384 : 8192) && p.n >= 1024 &&
         p.n < (1LL << 40) && p.n * p.k >= kStreamMinWeights;
}

int launch_stream(bool bf16, const GemmArgs& p, bool swiglu, bool norm, hipStream_t st) {
  if (bf16)
    launch_stream_d<bf16_t>(p, swiglu, norm, st);
  else
    launch_stream_d<half_t>(p, swiglu, norm, st);
  return check_launch("sph_gemm (stream)");
}

int launch_skinny(bool bf16, const GemmArgs& p, int64_t batch, bool norm, hipStream_t st) {
  if (bf16)
    norm ? skinny_t<bf16_t, true>(p, batch, st) : skinny_t<bf16_t, false>(p, batch, st);
  else
    norm ? skinny_t<half_t, true>(p, batch, st) : skinny_t<half_t, false>(p, batch, st);
  return check_launch("sph_gemm (small M)");
}

}  // namespace sph
