// The kernels that gemm.hip chooses from, by file.
#pragma once

#include "gemm_common.h"
#include "gemm_ring.h"

namespace sph {

// gemm_small.hip: at most 8 rows, K-contiguous operands.
constexpr int64_t kSmallRows = 8;
bool stream_fits(const GemmArgs& p, int64_t batch, bool a_kcont, bool b_kcont);
int launch_stream(bool bf16, const GemmArgs& p, bool swiglu, bool norm, hipStream_t st);
int launch_skinny(bool bf16, const GemmArgs& p, int64_t batch, bool norm, hipStream_t st);

// gemm_staged.hip: any layout, size and alignment.
int launch_staged(bool bf16, GemmArgs& p, int64_t batch, bool a_kcont, bool b_kcont,
                  hipStream_t st);

}  // namespace sph
