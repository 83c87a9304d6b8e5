// Plans and launches of the fp32 C = 32 and C = 64 kernels (nca_split_wide.h).
#include <hip/hip_runtime.h>

#include <string.h>

#include "nca_split_launch.h"
#include "nca_split_wide.h"

namespace nca {

namespace {

constexpr unsigned kWideLds = 160u * 1024u;
constexpr unsigned kSmallBytes = 4u * (256 + kSWN + 8 + 36);  // fc1's bias, fire factors, NaN flags, kernels

// LDS plan of R rows' rollout; false when it does not fit
bool wide_plan(int C, int R, int H, int W, int c_out, int n_out, SplitWide *sp) {
    const unsigned hw = (unsigned)H * W, hwp = (unsigned)(H + 2) * (W + 2);
    if ((uint64_t)R * hwp > 4096) return false;  // beyond any plan (and ci's 16 bits)
    sp->R = R;
    sp->l_Z = sp->l_red = 0;  // RED takes Z's place after fc1
    unsigned o = 2 * kSWZ;
    sp->l_small = o;
    o = st_al16(o + kSmallBytes);
    sp->l_P = o;
    o = st_al16(o + 2u * R * hwp * 4u * (C + 4));
    sp->l_ci = o;
    o = st_al16(o + 2u * R * hw);
    sp->l_fire = o;
    o = st_al16(o + 2u * R * hw);
    sp->l_given = o;
    o = st_al16(o + R * hw);
    sp->l_fired = o;
    o = st_al16(o + 4u * R);
    sp->l_head = o;
    o = st_al16(o + 4u * (n_out * c_out + n_out));
    sp->total = o;
    return o <= kWideLds;
}
static_assert(2 * kSWZ >= kSWRed, "RED in Z's place");

template <int C, bool GLOBAL, bool IN_NCHW, bool OUT_NCHW, int NT>
hipError_t launch(const SplitWide &sp, unsigned grid, hipStream_t st) {
    auto k = split_wide<C, GLOBAL, IN_NCHW, OUT_NCHW, NT>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)sp.total);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, dim3(grid), dim3(kSWT), sp.total, st, sp);
    return hipGetLastError();
}

template <int NT>
hipError_t launch_rollout(int C, const SplitWide &sp, unsigned grid, hipStream_t st) {
    return C == 32 ? launch<32, false, true, true, NT>(sp, grid, st) : launch<64, false, true, true, NT>(sp, grid, st);
}

}  // namespace

bool split_wide_resident_fits(int C, int H, int W, int c_out, int n_out) {
    SplitWide sp;
    return wide_plan(C, 1, H, W, c_out, n_out, &sp);
}

bool split_wide_step_fits(int C, int H, int W) {
    // a row within 31-bit byte offsets into the state
    return C == 32 && (int64_t)H * W * C * (int64_t)sizeof(float) < ((int64_t)1 << 31);
}

hipError_t split_wide_rollout(int C, const RolloutParams &p, hipStream_t st) {
    SplitWide sp;
    memset(&sp, 0, sizeof(sp));
    // the rows per workgroup and 32-cell tiles per pass with the least time on a CU: passes one after
    // another, of 6.2, 8.2 and 10.7 us (C = 32) or 10.7, 14.6 and 18.8 us (C = 64) for 1, 2 and 3 tiles. With
    // passes of 96 cells for every board, up to 256 boards of 5x5 took 10.8 and 18.8 us a step
    // where the fp32 MFMA kernel takes 10.0 and 16.8; 4,096 of 7x7 (C = 64) 320 where passes of 64 take 247.
    const int n_cu = plan_cus();
    int best = 0, nt = 0;
    int64_t cost = 0;
    for (int R = 1; R <= 16 && wide_plan(C, R, p.H, p.W, p.c_out, p.n_out, &sp); ++R) {
        const int64_t wgs = (p.rows + R - 1) / R, cells = (int64_t)R * p.H * p.W;
        for (int t = kSWNT; t >= 1; --t) {
            const int64_t c = ((wgs + n_cu - 1) / n_cu) * ((cells + 32 * t - 1) / (32 * t)) * (4 + 2 * t);
            if (!best || c < cost) best = R, nt = t, cost = c;
        }
    }
    if (!best || !wide_plan(C, best, p.H, p.W, p.c_out, p.n_out, &sp)) return hipErrorInvalidValue;
    sp.a = p;
    sp.wsplit = p.packed + p.off_split;
    const unsigned grid = (unsigned)((p.rows + best - 1) / best);
    if (nt == 1) return launch_rollout<1>(C, sp, grid, st);
    return nt == 2 ? launch_rollout<2>(C, sp, grid, st) : launch_rollout<3>(C, sp, grid, st);
}

hipError_t split_wide_step(const RolloutParams &p, int step, int first, int in_nchw, int out_nchw, hipStream_t st) {
    SplitWide sp;
    memset(&sp, 0, sizeof(sp));
    sp.wsplit = p.packed + p.off_split;
    sp.step = step;
    sp.first = first;
    sp.l_Z = 0;
    sp.l_red = 2 * kSWZ;
    sp.l_small = sp.l_red + kSWRed;
    sp.total = st_al16(sp.l_small + kSmallBytes);
    const int n_cu = plan_cus();
    const int64_t per = step_launch_rows(32, p.rows, p.H, p.W);
    for (int64_t r0 = 0; r0 < p.rows; r0 += per) {
        sp.a = step_rows(p, 32, step, r0, p.rows - r0 < per ? p.rows - r0 : per);
        sp.n_cells = (int)(sp.a.rows * p.H * p.W);
        sp.n_tiles = (sp.n_cells + kSWN - 1) / kSWN;
        sp.tiles_per_wg = (sp.n_tiles + n_cu - 1) / n_cu;
        const unsigned grid = (unsigned)((sp.n_tiles + sp.tiles_per_wg - 1) / sp.tiles_per_wg);
        const hipError_t e =
            in_nchw ? (out_nchw ? launch<32, true, true, true, kSWNT>(sp, grid, st) : launch<32, true, true, false, kSWNT>(sp, grid, st))
                    : (out_nchw ? launch<32, true, false, true, kSWNT>(sp, grid, st) : launch<32, true, false, false, kSWNT>(sp, grid, st));
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace nca
