// Entry points of the fp32 kernels on the bf16 matrix cores (nca_split.h).
#pragma once

#include <hip/hip_runtime.h>

#include "nca_rollout.h"

namespace nca {

// C = 16, 128 hidden units. A row's rollout in LDS (also recorded: x_rec, x_rec0); one step of rows
// of any size, x_in -> x_out (distinct buffers), in the caller's NCHW layout or cell-major, with
// 31-bit byte offsets into the state.
bool split16_resident_fits(int H, int W, int c_out, int n_out);
bool split16_step_fits(int64_t rows, int H, int W);
hipError_t split16_rollout(const RolloutParams &p, hipStream_t st);
hipError_t split16_step(const RolloutParams &p, int step, int first, int in_nchw, int out_nchw, hipStream_t st);

// C = 32 or 64, 256 hidden units: the same; the per-step kernel for C = 32 only.
bool split_wide_resident_fits(int C, int H, int W, int c_out, int n_out);
bool split_wide_step_fits(int C, int64_t rows, int H, int W);
hipError_t split_wide_rollout(int C, const RolloutParams &p, hipStream_t st);
hipError_t split_wide_step(const RolloutParams &p, int step, int first, int in_nchw, int out_nchw, hipStream_t st);

}  // namespace nca
