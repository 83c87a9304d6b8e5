// Plans and launches of the fp32 C = 16 kernels (nca_split16.h).
#include <hip/hip_runtime.h>

#include <string.h>

#include "nca_split16.h"
#include "nca_split_launch.h"

namespace nca {

namespace {

constexpr unsigned kSplitLds = 160u * 1024u;

// LDS plan for R rows; false when it does not fit
bool resident_plan(int R, int H, int W, int c_out, int n_out, Split16Resident *sp) {
    const unsigned hw = (unsigned)H * W, hwp = (unsigned)(H + 2) * (W + 2);
    if ((uint64_t)R * hwp > 4096) return false;  // beyond any plan (and ci's 16 bits)
    unsigned o = kSplit16Bytes + 512u;
    sp->R = R;
    sp->l_P = o;
    o = st_al16(o + 2u * R * hwp * 64u);
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
    return o <= kSplitLds;
}

template <bool IN_NCHW, bool OUT_NCHW>
hipError_t launch_step(const Split16Step &sp, unsigned grid, int first, hipStream_t st) {
    auto k = first ? step_split16<IN_NCHW, OUT_NCHW, true> : step_split16<IN_NCHW, OUT_NCHW, false>;
    constexpr unsigned lds = kSplit16Bytes + 512u;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, dim3(grid), dim3(kS16T), lds, st, sp);
    return hipGetLastError();
}

}  // namespace

bool split16_resident_fits(int H, int W, int c_out, int n_out) {
    Split16Resident sp;
    return resident_plan(1, H, W, c_out, n_out, &sp);
}

bool split16_step_fits(int H, int W) {
    // a row within 31-bit byte offsets into the cell-major state (cells past a row's end store at 2^31)
    return (int64_t)H * W * 16 * (int64_t)sizeof(float) < ((int64_t)1 << 31);
}

hipError_t split16_rollout(const RolloutParams &p, hipStream_t st) {
    Split16Resident sp;
    memset(&sp, 0, sizeof(sp));
    // enough rows per workgroup that a launch has about one workgroup per CU
    int R = (int)((p.rows + 255) / 256 < 16 ? (p.rows + 255) / 256 : 16);
    for (; R > 1 && !resident_plan(R, p.H, p.W, p.c_out, p.n_out, &sp); --R) {}
    if (!resident_plan(R, p.H, p.W, p.c_out, p.n_out, &sp)) return hipErrorInvalidValue;
    sp.a = p;
    sp.wsplit = p.packed + p.off_split;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(rollout_split16), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)sp.total);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(rollout_split16, dim3((unsigned)((p.rows + R - 1) / R)), dim3(kS16T), sp.total, st, sp);
    return hipGetLastError();
}

hipError_t split16_step(const RolloutParams &p, int step, int first, int in_nchw, int out_nchw, hipStream_t st) {
    Split16Step sp;
    memset(&sp, 0, sizeof(sp));
    sp.wsplit = p.packed + p.off_split;
    sp.step = step;
    sp.tiles_per_row = (p.H * p.W + 15) / 16;
    const int n_cu = plan_cus();
    const int64_t per = step_launch_rows(16, p.rows, p.H, p.W);
    for (int64_t r0 = 0; r0 < p.rows; r0 += per) {
        sp.a = step_rows(p, 16, step, r0, p.rows - r0 < per ? p.rows - r0 : per);
        sp.n_tiles = sp.a.rows * (int64_t)sp.tiles_per_row;
        sp.tiles_per_wg = (sp.n_tiles + n_cu - 1) / n_cu;
        const unsigned grid = (unsigned)((sp.n_tiles + sp.tiles_per_wg - 1) / sp.tiles_per_wg);
        const hipError_t e = in_nchw ? (out_nchw ? launch_step<true, true>(sp, grid, first, st) : launch_step<true, false>(sp, grid, first, st))
                                     : (out_nchw ? launch_step<false, true>(sp, grid, first, st) : launch_step<false, false>(sp, grid, first, st));
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace nca
