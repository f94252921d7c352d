// Ring-buffered GEMM for ragged and small row counts (gemm_ring.hip).
#pragma once

#include "gemm_common.h"

namespace sph {

struct RingPlan {
  int cfg = -1;        // tile configuration; -1: none fits
  int bm = 0, bn = 0;  // its tile
  int splits = 1;      // K slices
  int kslice = 0;      // K tiles per slice
  int64_t bytes = 0;   // workspace of the partial sums (0: one slice)
  double us = 0;       // modelled time
  double hot_us = 0;   // unsplit: time with operands in the caches (K up to ~1500)
};

// The fastest plan by the time model whose workspace is at most max_bytes.
RingPlan ring_plan(int64_t batch, int64_t m, int64_t n, int64_t k, bool b_kcont, bool swiglu,
                   int64_t max_bytes);

// What the kernel asks of a call: K-contiguous A, whole 16-byte chunks
// (K % 8, for row-major B nb % 8), 32-bit offsets.
bool ring_fits(const GemmArgs& p, bool a_kcont, bool b_kcont, bool swiglu);

// p.part must hold plan.bytes.
int launch_ring(bool bf16, GemmArgs& p, int64_t batch, bool b_kcont, bool swiglu,
                const RingPlan& plan, hipStream_t st);

}  // namespace sph
