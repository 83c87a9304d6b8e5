// Entry points of the fp32 kernels on the bf16 matrix cores (nca_split.h).
#pragma once

#include <hip/hip_runtime.h>

#include "nca_rollout.h"

namespace nca {

int device_cus();  // of the current device (nca_api.hip), 0 where it cannot be asked
inline int plan_cus() { return device_cus() > 0 ? device_cus() : 256; }

// C = 16, 128 hidden units. A row's rollout in LDS (also recorded: x_rec, x_rec0); one step of rows
// of any size, x_in -> x_out (distinct buffers), in the caller's NCHW layout or cell-major. The step
// kernels hold 31-bit byte offsets into the state: a launch takes as many rows as these reach, and
// a call's rows go in as many launches as they need, so that the choice of a kernel, and with it the
// rounding of a row, does not depend on the number of rows.
bool split16_resident_fits(int H, int W, int c_out, int n_out);
bool split16_step_fits(int H, int W);
hipError_t split16_rollout(const RolloutParams &p, hipStream_t st);
hipError_t split16_step(const RolloutParams &p, int step, int first, int in_nchw, int out_nchw, hipStream_t st);

// C = 32 or 64, 256 hidden units: the same; the per-step kernel for C = 32 only.
bool split_wide_resident_fits(int C, int H, int W, int c_out, int n_out);
bool split_wide_step_fits(int C, int H, int W);
hipError_t split_wide_rollout(int C, const RolloutParams &p, hipStream_t st);
hipError_t split_wide_step(const RolloutParams &p, int step, int first, int in_nchw, int out_nchw, hipStream_t st);

// Rows of a step launch: the call's rows in equal parts whose states stay below 2 GiB.
inline int64_t step_launch_rows(int C, int64_t rows, int H, int W) {
    const int64_t most = (((int64_t)1 << 31) - 1) / ((int64_t)C * H * W * (int64_t)sizeof(float));
    const int64_t parts = (rows + most - 1) / most;
    return parts > 1 ? (rows + parts - 1) / parts : rows;
}

// Rows [r0, r0 + n) of step `step` of a call; fire_u8 is that step's masks.
inline RolloutParams step_rows(const RolloutParams &p, int C, int step, int64_t r0, int64_t n) {
    RolloutParams q = p;
    const int64_t hw = (int64_t)p.H * p.W;
    q.rows = n;
    q.row0 = p.row0 + r0;
    q.x_in = p.x_in + r0 * C * hw;
    q.x_out = p.x_out + r0 * C * hw;
    q.given = p.given + r0 * hw;
    if (p.clamp) q.clamp = p.clamp + r0 * p.c_in * hw;
    if (p.noise) q.noise = p.noise + r0 * C * hw;
    if (p.fire_f32) q.fire_f32 = p.fire_f32 + r0 * hw;
    if (p.fire_u8) q.fire_u8 = p.fire_u8 + (step * p.rows + r0) * hw;
    if (p.fired_out) q.fired_out = p.fired_out + r0;
    return q;
}

}  // namespace nca
