// fp32 cells with 256 hidden units and C = 32 or 64 channels (gfx950), on the bf16 matrix cores with
// operands in three bf16 parts (nca_split.h): one step of boards of any size per launch (GLOBAL,
// C = 32), and the rollout of boards that fit the LDS in one launch.
//
// The weights' three parts (240 KB at C = 32, 480 KB at C = 64) fit neither LDS nor, beside the
// accumulators, the registers: they stream from L2 and are shared by a pass of up to 96 cells. Each of 8
// waves owns 32 hidden units of all its cells (three 32x32 accumulator tiles), so that a weight
// fragment is loaded once per pass and workgroup and used for three products, and its loads for
// the k-step after next are issued as a step's are used. Per interval of 64 features (16
// channels, 4 kernels) and one barrier, the waves multiply one half of Z (LDS, three parts) while
// they compute the other from the taps: v_mfma_f32_32x32x16_bf16 leaves the issue port to the
// stencil. fc1's accumulators are fc2's B operand as they lie; the 8 partial sums of dx meet in LDS
// (RED) and are added in one order. The largest products and the five smaller ones have sums of
// their own (a rounding of a smaller sum costs less).
//
// Per 16 cells and CU the MFMAs take 1,920 (C = 32) or 3,840 cycles; they are busy for 49 % of the
// time at C = 64 and 35 % at C = 32. What is left, from versions without each part (64 steps of
// 2,048 boards 9x9 / 32 steps of 512 boards 30x30, fp32): fc1's products alone 6.3 / 4.4 ms, with the
// stencil 7.9 / 5.4, with fc2 and the update but no stencil 9.6 / 6.9. The registers are full (96 of
// 256 are fc1's accumulators): what splits a wave's code by a branch (waves without a stencil, half
// of the waves updating while the others multiply) spilled 200 of them and took twice as long.
// Measured against the fp32 MFMA kernels: 2,048 boards 9x9, 64 steps 21.2 -> 10.1 to 10.7 ms; 512
// boards 30x30, gated, 32 steps 14.9 -> 8.4 to 9.5 ms by box; error against 64 bits of a step 0.3 to 0.4 of theirs.
#pragma once

#include "nca_split.h"

namespace nca {

constexpr int kSWT = 512;                       // threads per workgroup: 8 waves
constexpr int kSWN = 96, kSWNT = 3;             // most cells of a pass, 32-cell tiles
constexpr int kSWStride = 98;                   // 16-byte units between Z's (quad, half) planes: 4 quads x
                                                // 4 cells fall on distinct LDS slots
constexpr unsigned kSWZ = 3u * 4u * 2u * kSWStride * 16u;  // bytes of one Z buffer: [part][quad][half][cell]
constexpr unsigned kSWRed = 65536u;             // RED: [wave][channel quad][cell], 32 or 64 cells at a time

struct SplitWide {
    RolloutParams a;
    const unsigned char *wsplit;
    int step, first;            // per-step launches: step index within the call, first step of the call
                                // (a.fire_u8: the step's masks)
    int n_cells, n_tiles, tiles_per_wg;
    int R;                      // rollouts in LDS: rows per workgroup
    unsigned l_Z, l_red, l_small, l_P, l_ci, l_fire, l_given, l_fired, l_head, total;
};

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma32(uint4 a, uint4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// GLOBAL: one step, the state in global memory (cell-major, or the caller's NCHW); otherwise R rows'
// whole rollout in LDS, the state twice (a step reads one, writes the other), with a one-cell border.
// A pass takes NT tiles: a workgroup with few cells would spend a pass of three on nothing (their
// cells' bits are the same in every form).
template <int C, bool GLOBAL, bool IN_NCHW, bool OUT_NCHW, int NT>
__global__ void __launch_bounds__(kSWT, 1) split_wide(SplitWide sp) {
    constexpr int PN = 32 * NT;  // cells of a pass
    constexpr int HD = 256, KS = C / 16, MT = C / 32, NQ = C / 4, CP = C + 4;
    constexpr int NTR = 64 / C;  // 32-cell tiles of a reduction round: 512 (cell, quad) items
    const RolloutParams &a = sp.a;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *Zb = smem + sp.l_Z;
    float4 *RED = reinterpret_cast<float4 *>(smem + sp.l_red);
    float *b1L = reinterpret_cast<float *>(smem + sp.l_small);
    float *fireG = b1L + HD;                                // GLOBAL: fire factors of the pass's cells
    // the cells of each 32-cell tile with a NaN among their sums, a bit each, for even and odd passes: a
    // pass clears the other's after its first barrier, when every wave is past the last look at them
    int *badL = reinterpret_cast<int *>(fireG + PN), *bad = badL;
    f32x4 *kernL = reinterpret_cast<f32x4 *>(badL + 8);      // the 4 kernels' weights of each tap
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, hf = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, W = a.W, HWn = H * W;
    const float *padv = reinterpret_cast<const float *>(a.packed + a.off_padv);
    const bool wrap = a.padding == 2;
    const int c_in = a.c_in, in_off = a.in_off;
    for (int e = tid; e < HD; e += kSWT) b1L[e] = reinterpret_cast<const float *>(a.packed + a.off_b1)[e];
    if (tid < 8) badL[tid] = 0;
    if (tid < 36) reinterpret_cast<float *>(kernL)[tid] = reinterpret_cast<const float *>(a.packed + a.off_kern)[(tid & 3) * 9 + (tid >> 2)];
    __syncthreads();

    // ---- the rollout's LDS state
    float *P = reinterpret_cast<float *>(smem + sp.l_P);
    uint16_t *ci = reinterpret_cast<uint16_t *>(smem + sp.l_ci);  // cell -> bordered cell
    uint8_t *fireL = smem + sp.l_fire, *givenL = smem + sp.l_given;
    int *firedL = reinterpret_cast<int *>(smem + sp.l_fired);
    float *headL = reinterpret_cast<float *>(smem + sp.l_head);
    const int Wp = W + 2, HWp = (H + 2) * Wp;
    const int64_t rbase = GLOBAL ? 0 : (int64_t)blockIdx.x * sp.R;
    const int Rw = GLOBAL ? 0 : (int)(a.rows - rbase < sp.R ? a.rows - rbase : sp.R);
    const int ncell = GLOBAL ? sp.n_cells : Rw * HWn, PB = sp.R * HWp * CP;
    int cur = 0;

    // ---- taps of (cell gq, channel quad cq)
    // the position of a cell's taps: clamped to the last cell past the end
    struct Pos {
        int base, ro0, ro2, co0, co2, padm, row, q;
    };
    auto locate = [&](int gq) __attribute__((always_inline)) {
        Pos p;
        const int gc = gq < ncell ? gq : ncell - 1;
        if constexpr (GLOBAL) {
            p.row = (int)((unsigned)gc / (unsigned)HWn);
            p.q = gc - p.row * HWn;
            const int i = (int)((unsigned)p.q / (unsigned)W), j = p.q - i * W;
            p.base = gc;
            p.ro0 = i > 0 ? -W : (H - 1) * W;
            p.ro2 = i < H - 1 ? W : -(H - 1) * W;
            p.co0 = j > 0 ? -1 : W - 1;
            p.co2 = j < W - 1 ? 1 : -(W - 1);
            p.padm = wrap ? 0
                          : ((i == 0 ? 0x007 : 0) | (i == H - 1 ? 0x1c0 : 0) | (j == 0 ? 0x049 : 0) |
                             (j == W - 1 ? 0x124 : 0));
        } else {
            p.base = ci[gc] * CP;
            p.padm = 0;
        }
        return p;
    };
    auto load_tap = [&](const Pos &p, int cq, int t) __attribute__((always_inline)) {
        if constexpr (GLOBAL) {
            const int d = (t < 3 ? p.ro0 : t < 6 ? 0 : p.ro2) + (t % 3 == 0 ? p.co0 : t % 3 == 1 ? 0 : p.co2);
            if (IN_NCHW) {
                const float *xr = a.x_in + ((int64_t)p.row * C + 4 * cq) * HWn + p.q + d;
                return f32x4{xr[0], xr[HWn], xr[2 * HWn], xr[3 * HWn]};
            }
            const uint32_t off = (uint32_t)(p.base + d) * (uint32_t)(4 * C) + 16u * (uint32_t)cq;
            return *reinterpret_cast<const f32x4 *>(reinterpret_cast<const unsigned char *>(a.x_in) + off);
        } else {
            return *reinterpret_cast<const f32x4 *>(P + cur * PB + p.base + 4 * cq + ((t / 3 - 1) * Wp + t % 3 - 1) * CP);
        }
    };
    // z += kernel weights of tap t x its value (stencil16's chains)
    auto add_tap = [&](const Pos &p, f32x4 pq, f32x4 tp, f32x4 kw, int t, float z[4][4]) __attribute__((always_inline)) {
        const bool o = GLOBAL && t != 4 && ((p.padm >> t) & 1);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float v = o ? pq[c] : tp[c];
#pragma unroll
            for (int k = 0; k < 4; ++k) z[k][c] = __builtin_fmaf(kw[k], v, t == 0 ? 0.0f : z[k][c]);
        }
    };
    auto pad_quad = [&](int cq) __attribute__((always_inline)) {
        return GLOBAL && a.padding == 1 ? reinterpret_cast<const f32x4 *>(padv)[cq] : f32x4{0.f, 0.f, 0.f, 0.f};
    };

    // the stencil item of a thread: cell sc, quad sq of an interval's 4. Quads fastest for global loads
    // (64 bytes of a cell), cells fastest for LDS taps (an odd stride of 16-byte slots). Waves 6 and 7
    // repeat waves 0 and 1's: a branch here doubles the intervals' code and spills the accumulators.
    const int sid = tid % (4 * PN);
    const int sc = GLOBAL ? sid >> 2 : 16 * (sid >> 6) + (sid & 15), sq = GLOBAL ? sid & 3 : (sid >> 4) & 3;
    auto put_half = [&](const float z[4][4], int h, int buf) __attribute__((always_inline)) {
        uint4 *zp = reinterpret_cast<uint4 *>(Zb + buf * kSWZ) + (2 * sq + h) * kSWStride + sc;
        const float v[8] = {z[2 * h][0],     z[2 * h][1],     z[2 * h][2],     z[2 * h][3],
                            z[2 * h + 1][0], z[2 * h + 1][1], z[2 * h + 1][2], z[2 * h + 1][3]};
        const Split8 s = split8(v);
        zp[0] = s.h;
        zp[8 * kSWStride] = s.m;
        zp[16 * kSWStride] = s.l;
    };
    auto stencil_quad = [&](const Pos &p, int cq, float z[4][4]) __attribute__((always_inline)) {
        f32x4 tp[9];
        const f32x4 pq = pad_quad(cq);
#pragma unroll
        for (int t = 0; t < 9; ++t) tp[t] = load_tap(p, cq, t);
#pragma unroll
        for (int t = 0; t < 9; ++t) add_tap(p, pq, tp[t], kernL[t], t, z);
    };
    auto put_z = [&](const Pos &p) __attribute__((always_inline)) {  // the first interval's
        float z[4][4];
        stencil_quad(p, sq, z);
        put_half(z, 0, 0);
        put_half(z, 1, 0);
    };

    // ---- weight fragments: W1 [wave][k-step C][part][lane], W2 [wave][m-tile][k-step 2][part][lane]
    // through a buffer descriptor: the fragment's place is a scalar offset, no address per lane
    constexpr unsigned kWA = 8u * (C / 4) * 3072u, kWB = 8u * MT * 2 * 3072u;
    const __amdgpu_buffer_rsrc_t w_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char *>(sp.wsplit), (short)0, (int)(kWA + kWB), 0x00020000);
    const unsigned wA = (unsigned)w * (C / 4) * 3072u, wB = kWA + (unsigned)w * MT * 2 * 3072u;
    auto frag = [&](unsigned base, int f) __attribute__((always_inline)) {
        auto ld = [&](unsigned part) __attribute__((always_inline)) {
            return __builtin_bit_cast(
                uint4, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, 16u * lane, base + (unsigned)f * 3072u + part * 1024u, 0));
        };
        return Split8{ld(0), ld(1), ld(2)};
    };
    Split8 af[2] = {frag(wA, 0), frag(wA, 1)};

    // ---- one pass: cells [g0, g0 + 32 NT) of step s (its index in the call)
    const float4 b2v = reinterpret_cast<const float4 *>(a.packed + a.off_b2)[tid / (32 * NTR)];
    // GLOBAL: waves 6 and 7 draw the fire factors of the pass's cells. What they read is touched an
    // interval earlier.
    auto warm_fire = [&](int g0) __attribute__((always_inline)) {
        const int k = tid & 127, gc = k < PN && g0 + k < ncell ? g0 + k : g0;
        float v = (float)a.given[gc];
        if (a.adaptive && !IN_NCHW) v += a.x_in[(int64_t)gc * C + a.out_off];
        return v;
    };
    auto draw_pass = [&](int g0) __attribute__((always_inline)) {
        const int k = tid - 384, gq = g0 + k;
        const bool live = k < PN && gq < ncell;
        const int gc = live ? gq : g0, row = (int)((unsigned)gc / (unsigned)HWn), q = gc - row * HWn;
        float f;
        if (a.fire_f32) {
            f = a.fire_f32[gc];
        } else if (a.fire_u8) {
            f = a.fire_u8[gc] ? 1.0f : 0.0f;
        } else {
            const uint64_t key = a.step_seeds ? a.step_seeds[sp.step] : a.seed;
            float u4[4];
            cell_uniforms4(key, (uint32_t)(a.row0 + row), (uint32_t)(a.step0 + sp.step), (uint32_t)(q >> 2), u4);
            const float u = (q & 3) == 0 ? u4[0] : (q & 3) == 1 ? u4[1] : (q & 3) == 2 ? u4[2] : u4[3];
            float p = a.p;
            if (a.adaptive) {
                const float *hw = reinterpret_cast<const float *>(a.packed + a.off_headw);
                const float *hb = reinterpret_cast<const float *>(a.packed + a.off_headb);
                int am;
                const float *xc = IN_NCHW ? a.x_in + ((int64_t)row * C + a.out_off) * HWn + q : a.x_in + (int64_t)gc * C + a.out_off;
                const float cf = cell_readout(xc, IN_NCHW ? HWn : 1, a.c_out, a.n_out, a.head_kind, hw, hb, &am);
                if (cf > a.tau || (a.given_confident && a.given[gc])) p = a.p_low;
            }
            f = u < p ? 1.0f : 0.0f;
        }
        if (k < PN) fireG[k] = f;
        if (a.fired_out) {
            // one addition per row of the wave's cells
            uint64_t rest = __ballot(live && f != 0.0f);
            while (rest) {
                const int r0 = __builtin_amdgcn_readlane(row, (int)__builtin_ctzll(rest));
                const uint64_t mine = __ballot(live && f != 0.0f && row == r0);
                if (lane == 0) atomicAdd(a.fired_out + r0, (int)__popcll(mine));
                rest &= ~mine;
            }
        }
    };
    auto pass = [&](int g0, int g0_next, int s, bool first, Pos &pos) __attribute__((always_inline)) {
        f32x16 big[NT], small[NT];
        auto bias = [&]() __attribute__((always_inline)) {
            f32x16 r;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float4 b = *reinterpret_cast<const float4 *>(b1L + 32 * w + 8 * v + 4 * hf);
                r[4 * v] = b.x, r[4 * v + 1] = b.y, r[4 * v + 2] = b.z, r[4 * v + 3] = b.w;
            }
            return r;
        };
        const f32x16 b1v = bias();
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            big[t] = b1v;
            small[t] = f32x16{};
        }
        // An interval is 12 steps: per 16 features the l, m and h parts of Z, each with the weight parts
        // it meets. A step's fragments are read two steps ahead; the steps between
        // also add the taps into the next interval's z, which the last two split and store. Taps from
        // global memory are loaded in the first three steps and added from the third on (later, at about 2,000
        // cycles, they hold registers for longer: 30x30 steps 5 % slower), taps from LDS two steps ahead.
        // The barriers for the scheduler keep the loads where they are.
        auto interval = [&](int i, const Pos &ps, int cq, int next, auto with_stencil) __attribute__((always_inline)) {
            constexpr bool ST = decltype(with_stencil)::value;
            const uint4 *zb = reinterpret_cast<const uint4 *>(Zb + (i & 1) * kSWZ) + hf * kSWStride + n;
            uint4 v[3][NT];
            constexpr int NTP = GLOBAL ? 9 : 4;
            f32x4 tp[NTP], pq;
            float z[4][4];
            auto load_v = [&](int st) __attribute__((always_inline)) {
#pragma unroll
                for (int t = 0; t < NT; ++t) v[st % 3][t] = zb[((2 - st % 3) * 8 + 2 * (st / 3)) * kSWStride + 32 * t];
            };
            load_v(0);
            load_v(1);
            if constexpr (ST) pq = pad_quad(cq);
#pragma unroll
            for (int st = 0; st < 12; ++st) {
                __builtin_amdgcn_sched_barrier(0);
                const int j = st / 3;
                if (st + 2 < 12) load_v(st + 2);
                if constexpr (ST) {
#pragma unroll
                    for (int t = 0; t < 9; ++t)
                        if (st == (GLOBAL ? t / 3 : t > 1 ? t - 1 : 0)) tp[t % NTP] = load_tap(ps, cq, t);
                }
                const Split8 &wf = af[j & 1];
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    if (st % 3 == 2)
                        big[t] = mfma32(wf.h, v[2][t], big[t]);
                    else
                        small[t] = mfma32(wf.h, v[st % 3][t], small[t]);
                }
                if (st % 3 >= 1) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) small[t] = mfma32(wf.m, v[st % 3][t], small[t]);
                }
                if (st % 3 == 2) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) small[t] = mfma32(wf.l, v[2][t], small[t]);
                    af[j & 1] = frag(wA, j < 2 ? 4 * i + j + 2 : 4 * next + j - 2);
                }
                if constexpr (ST) {
#pragma unroll
                    for (int t = 0; t < 9; ++t)
                        if (st == (GLOBAL ? 2 + t : 1 + t)) add_tap(ps, pq, tp[t % NTP], kernL[t], t, z);
                    if (st == 10) put_half(z, 0, (i + 1) & 1);
                    if (st == 11) put_half(z, 1, (i + 1) & 1);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll 1
        for (int i = 0; i + 1 < KS; ++i) {
            const float warm = GLOBAL ? warm_fire(g0) : 0.0f;
            interval(i, pos, 4 * (i + 1) + sq, i + 1, std::true_type{});
            if constexpr (GLOBAL) {
                asm volatile("" ::"v"(warm));
                if (i == 0 && w >= 6) draw_pass(g0);
            }
            __syncthreads();
            if (tid < 4) badL[(bad == badL ? 4 : 0) + tid] = 0;
        }
        if constexpr (GLOBAL) pos = locate(g0_next + sc);
        interval(KS - 1, pos, sq, 0, std::integral_constant<bool, GLOBAL>{});

        // ---- fc2 and the update, a round of NTR 32-cell tiles after another: the partial sums of a
        // round meet in RED between two barriers; a round's update runs beside the next one's products
        constexpr int RC = 32 * NTR, NR = (NT + NTR - 1) / NTR;
        const int ic = tid % RC, iq = tid / RC;  // this thread's item of a round: cell, channel quad
        Split8 wf[MT][2];
        bool nanh[2][NTR];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) wf[mt][0] = frag(wB, 2 * mt), wf[mt][1] = frag(wB, 2 * mt + 1);
        f32x16 part[NTR][MT];
        Split8 hs[2][NTR][2];
        // h of the round's tiles in three parts, as the products' B operands; round rd's in hs[rd & 1]
        auto split_h = [&](int rd) __attribute__((always_inline)) {
#pragma unroll
            for (int tr = 0; tr < NTR; ++tr) {
                const int t = rd * NTR + tr;
                if (t >= NT) break;
                const f32x16 h = big[t] + small[t];
                bool nan = false;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    float hv[8];
#pragma unroll
                    for (int v = 0; v < 8; ++v) hv[v] = relu_f32(h[8 * j + v]);
#pragma unroll
                    for (int v = 0; v < 8; v += 2) nan |= __builtin_isunordered(h[8 * j + v], h[8 * j + v + 1]);
                    hs[rd & 1][tr][j] = split8(hv);
                }
                nanh[rd & 1][tr] = nan;
            }
        };
        auto products = [&](int rd) __attribute__((always_inline)) {
            // the smaller products first: the sums are full-size for the last two only
#pragma unroll
            for (int tr = 0; tr < NTR; ++tr)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) part[tr][mt] = f32x16{};
            auto add = [&](auto pw, auto ph) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int tr = 0; tr < NTR; ++tr)
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt)
                            if (rd * NTR + tr < NT)
                                part[tr][mt] = mfma32(wf[mt][j].*pw, hs[rd & 1][tr][j].*ph, part[tr][mt]);
            };
            add(&Split8::l, &Split8::h);
            add(&Split8::h, &Split8::l);
            add(&Split8::m, &Split8::m);
            add(&Split8::m, &Split8::h);
            add(&Split8::h, &Split8::m);
            add(&Split8::h, &Split8::h);
        };
        // marks cells with a NaN among h
        auto mark = [&](int rd) __attribute__((always_inline)) {
#pragma unroll
            for (int tr = 0; tr < NTR; ++tr) {
                if (rd * NTR + tr >= NT) break;
                const uint64_t m = __ballot(nanh[rd & 1][tr]);
                if (m && lane == 0) atomicOr(&bad[rd * NTR + tr], (int)(m | m >> 32));
            }
        };
        // one MFMA, then VALU work beside it
        auto mix = [&](int mfmas) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < 24; ++k)
                if (k < mfmas) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
                }
        };
        auto put_part = [&](int tr, int mt, f32x16 d) __attribute__((always_inline)) {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                RED[(w * NQ + 8 * mt + 2 * v + hf) * RC + 32 * tr + n] =
                    make_float4(d[4 * v], d[4 * v + 1], d[4 * v + 2], d[4 * v + 3]);
        };
        // the update of the round's items: the sums from RED and the new state, without a branch, then the
        // rest; a NaN of dx marks its cell. again: only the marked cells
        auto sums = [&](f32x4 xo, int gv, float f, f32x4 &u) __attribute__((always_inline)) {
            float4 r[8];
#pragma unroll
            for (int k8 = 0; k8 < 8; ++k8) r[k8] = RED[(k8 * NQ + iq) * RC + ic];
            f32x4 dx;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                auto e = [&](int k8) { return (&r[k8].x)[v]; };
                dx[v] = __fadd_rn(__fadd_rn(__fadd_rn(__fadd_rn(e(0), e(1)), __fadd_rn(e(2), e(3))),
                                            __fadd_rn(__fadd_rn(e(4), e(5)), __fadd_rn(e(6), e(7)))),
                                  (&b2v.x)[v]);
                const int c = 4 * iq + v;
                const float uv = __fadd_rn(xo[v], __fmul_rn(f, dx[v]));
                u[v] = (gv != 0) & (c >= in_off) & (c < in_off + c_in) ? xo[v] : uv;
            }
            return __builtin_isunordered(dx[0], dx[1]) | __builtin_isunordered(dx[2], dx[3]);
        };
        auto finish = [&](int t0, f32x4 u, int gv, float f, bool nan, bool again) __attribute__((always_inline)) {
            const int k = 32 * t0 + ic, gq = g0 + k;
            bool live = gq < ncell && k < PN;
            const int gc = live ? gq : g0;
            if (again) {
                live = live && ((bad[t0 + (ic >> 5)] >> (ic & 31)) & 1);
            } else if (const uint64_t m = __ballot(live && nan); m && lane == 0) {
                // a wave's lanes are the round's 64 cells, or two quads of its 32
                if (NTR > 1) {
                    atomicOr(&bad[t0], (int)m);
                    if (t0 + 1 < NT) atomicOr(&bad[t0 + 1], (int)(m >> 32));
                } else {
                    atomicOr(&bad[t0], (int)(m | m >> 32));
                }
            }
            if (a.noise || (first && c_in > 0) || (!GLOBAL && (a.x_rec || a.fire_f32)) || (GLOBAL && OUT_NCHW)) {
                const int row = (int)((unsigned)gc / (unsigned)HWn), q = gc - row * HWn;
                const int64_t grow = rbase + row;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int c = 4 * iq + v;
                    const bool frozen = (gv != 0) & (c >= in_off) & (c < in_off + c_in);
                    if (a.noise && !frozen) u[v] = __fadd_rn(u[v], a.noise[(grow * C + c) * HWn + q]);
                    if (first && frozen) u[v] = a.clamp[(grow * c_in + c - in_off) * HWn + q];
                }
                float *xr = nullptr;
                if (GLOBAL && OUT_NCHW) xr = a.x_out;
                if (!GLOBAL && a.x_rec) xr = a.x_rec + s * a.rec_stride;
                if (xr && live) {
                    xr += (grow * C + 4 * iq) * HWn + q;
#pragma unroll
                    for (int v = 0; v < 4; ++v) xr[(int64_t)v * HWn] = u[v];
                }
                if (!GLOBAL && a.fire_f32 && !again && live && iq == 0 && f != 0.0f) atomicAdd(&firedL[row], 1);
            }
            if (!live) return;
            if constexpr (!GLOBAL)
                *reinterpret_cast<f32x4 *>(P + (cur ^ 1) * PB + ci[gc] * CP + 4 * iq) = u;
            else if constexpr (!OUT_NCHW)
                *reinterpret_cast<f32x4 *>(a.x_out + (int64_t)gc * C + 4 * iq) = u;
        };
        // what the update of this thread's item reads besides
        auto load_item = [&](int t0, f32x4 &xo, int &gv, float &f) __attribute__((always_inline)) {
            const int k = 32 * t0 + ic, gq = g0 + k;
            const bool live = gq < ncell && k < PN;
            const int gc = live ? gq : g0;
            if constexpr (GLOBAL) {
                if (IN_NCHW) {
                    const int row = (int)((unsigned)gc / (unsigned)HWn), q = gc - row * HWn;
                    const float *xr = a.x_in + ((int64_t)row * C + 4 * iq) * HWn + q;
                    xo = f32x4{xr[0], xr[HWn], xr[2 * HWn], xr[3 * HWn]};
                } else {
                    xo = *reinterpret_cast<const f32x4 *>(a.x_in + (int64_t)gc * C + 4 * iq);
                }
                gv = a.given[gc];
                f = fireG[live ? k : 0];
            } else {
                xo = *reinterpret_cast<const f32x4 *>(P + cur * PB + ci[gc] * CP + 4 * iq);
                gv = givenL[gc];
                f = a.fire_f32 ? a.fire_f32[rbase * HWn + gc] : fireL[(s & 1) * sp.R * HWn + gc] ? 1.0f : 0.0f;
            }
        };
        // a NaN among a round's sums: its tiles on fp32 MFMA (z through RED, feature-major), whose result the
        // marked cells take
        auto redo = [&](int t0) {
            const int k = 32 * t0 + ic, gq = g0 + k;
            const int gc = gq < ncell && k < PN ? gq : g0;
            float *zf = reinterpret_cast<float *>(RED);
            const float *w1f = reinterpret_cast<const float *>(a.packed + a.off_w1);
            const float *w2f = reinterpret_cast<const float *>(a.packed + a.off_w2);
            asm volatile("" : "+s"(w1f), "+s"(w2f));  // addresses formed here, not kept across the passes
            {
                const Pos p = locate(gc);
                float z[4][4];
                stencil_quad(p, iq, z);
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                    for (int c = 0; c < 4; ++c) zf[(kk * C + 4 * iq + c) * RC + ic] = z[kk][c];
            }
            __syncthreads();
            f32x16 pt[NTR][MT];
#pragma unroll
            for (int tr = 0; tr < NTR; ++tr) {
                f32x16 h = bias();
#pragma unroll 1
                for (int kk = 0; kk < 4 * C; kk += 2) {
                    const float av = w1f[(((2 * w + (n >> 4)) * (C / 4) + (kk >> 4)) * 64 + ((kk & 3) + hf) * 16 + (n & 15)) * 4 + ((kk >> 2) & 3)];
                    h = __builtin_amdgcn_mfma_f32_32x32x2f32(av, zf[(kk + hf) * RC + 32 * tr + n], h, 0, 0, 0);
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    f32x16 d = f32x16{};
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int hid = 32 * w + 8 * (v / 4) + 4 * hf + v % 4, m = 32 * mt + n;
                        const float av = w2f[((m >> 4) * (HD / 4) + (hid >> 2)) * 64 + (hid & 3) * 16 + (m & 15)];
                        d = __builtin_amdgcn_mfma_f32_32x32x2f32(av, h[v] > 0.0f ? h[v] : 0.0f, d, 0, 0, 0);
                    }
                    pt[tr][mt] = d;
                }
            }
            __syncthreads();
#pragma unroll
            for (int tr = 0; tr < NTR; ++tr)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) put_part(tr, mt, pt[tr][mt]);
            __syncthreads();
            f32x4 xo, u;
            int gv;
            float f;
            load_item(t0, xo, gv, f);
            sums(xo, gv, f, u);
            finish(t0, u, gv, f, false, true);
            __syncthreads();
        };
        // the global ones of all rounds now, ahead of their use
        f32x4 xo[NR];
        int gv[NR];
        float f[NR];
        if constexpr (GLOBAL) {
#pragma unroll
            for (int rd = 0; rd < NR; ++rd) load_item(rd * NTR, xo[rd], gv[rd], f[rd]);
        }
        split_h(0);
        __builtin_amdgcn_sched_barrier(0);
        products(0);
        if (NR > 1) split_h(1);
        mix(12 * NTR * MT);
        __builtin_amdgcn_sched_barrier(0);
        mark(0);
        __syncthreads();  // Z's last half is read (RED may take its place)
#pragma unroll
        for (int rd = 0; rd < NR; ++rd) {
            const int t0 = rd * NTR;
#pragma unroll
            for (int tr = 0; tr < NTR; ++tr)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    if (t0 + tr < NT) put_part(tr, mt, part[tr][mt]);
            if constexpr (!GLOBAL) load_item(t0, xo[rd], gv[rd], f[rd]);
            __syncthreads();
            f32x4 u;
            __builtin_amdgcn_sched_barrier(0);
            if (rd + 1 < NR) products(rd + 1);
            const bool nan = sums(xo[rd], gv[rd], f[rd], u);
            if (rd + 2 < NR) split_h(rd + 2);
            if (rd + 1 < NR) mix(12 * NTR * MT);
            __builtin_amdgcn_sched_barrier(0);
            if (rd + 1 < NR) mark(rd + 1);
            finish(t0, u, gv[rd], f[rd], nan, false);
            __syncthreads();
            bool any = bad[t0] != 0;
            if (NTR > 1 && t0 + 1 < NT) any |= bad[t0 + 1] != 0;
            if (__builtin_amdgcn_readfirstlane(any)) redo(t0);
        }
        bad = bad == badL ? badL + 4 : badL;
    };

    if constexpr (GLOBAL) {
        const int t_begin = (int)blockIdx.x * sp.tiles_per_wg;
        const int t_end = t_begin + sp.tiles_per_wg < sp.n_tiles ? t_begin + sp.tiles_per_wg : sp.n_tiles;
        Pos pos = locate(t_begin * PN + sc);
        put_z(pos);
        __syncthreads();
        for (int t = t_begin; t < t_end; ++t) {
            const int g0 = t * PN;
            pass(g0, t + 1 < t_end ? g0 + PN : g0, sp.step, sp.first != 0, pos);
        }
    } else {
        // ---- the rows' state, given flags and cell table; the constant border
        for (int e = tid; e < Rw * C * HWn; e += kSWT) {
            const int rr = e / (C * HWn), rem = e - rr * C * HWn, c = rem / HWn, q = rem - c * HWn;
            const float v = a.x_in[rbase * C * HWn + e];
            P[(rr * HWp + (q / W + 1) * Wp + q % W + 1) * CP + c] = v;
            if (a.x_rec0) a.x_rec0[rbase * C * HWn + e] = v;
        }
        for (int e = tid; e < ncell; e += kSWT) {
            const int rr = e / HWn, q = e - rr * HWn;
            givenL[e] = a.given[rbase * HWn + e];
            ci[e] = (uint16_t)(rr * HWp + (q / W + 1) * Wp + q % W + 1);
        }
        for (int e = tid; e < sp.R; e += kSWT) firedL[e] = 0;
        {
            const float *hw = reinterpret_cast<const float *>(a.packed + a.off_headw);
            const float *hb = reinterpret_cast<const float *>(a.packed + a.off_headb);
            const int nw = a.n_out * a.c_out;
            for (int e = tid; e < nw + a.n_out; e += kSWT) headL[e] = e < nw ? hw[e] : hb[e - nw];
        }
        const int nhalo = 2 * Wp + 2 * H;
        auto halo_cell = [&](int h, int &ip, int &jp) {
            if (h < 2 * Wp) {
                ip = h < Wp ? 0 : H + 1;
                jp = h < Wp ? h : h - Wp;
            } else {
                ip = (h - 2 * Wp) % H + 1;
                jp = h - 2 * Wp < H ? 0 : W + 1;
            }
        };
        if (!wrap)
            for (int e = tid; e < 2 * Rw * nhalo * C; e += kSWT) {
                const int c = e % C, rest = e / C, h = rest % nhalo, rb = rest / nhalo, rr = rb % Rw, buf = rb / Rw;
                int ip, jp;
                halo_cell(h, ip, jp);
                P[buf * PB + (rr * HWp + ip * Wp + jp) * CP + c] = a.padding == 1 ? padv[c] : 0.0f;
            }
        auto wrap_halo = [&](int buf) {
            for (int e = tid; e < Rw * nhalo * NQ; e += kSWT) {
                const int qd = e % NQ, rest = e / NQ, h = rest % nhalo, rr = rest / nhalo;
                int ip, jp;
                halo_cell(h, ip, jp);
                const int si = ip == 0 ? H : ip == H + 1 ? 1 : ip, sj = jp == 0 ? W : jp == W + 1 ? 1 : jp;
                float *p = P + buf * PB + rr * HWp * CP + 4 * qd;
                *reinterpret_cast<float4 *>(p + (ip * Wp + jp) * CP) = *reinterpret_cast<const float4 *>(p + (si * Wp + sj) * CP);
            }
        };
        // fire bytes of step s (the state in buffer b is the step's input) into half s & 1
        const int nq = (HWn + 3) >> 2;
        auto draw_fire = [&](int s, int b) {
            if (a.fire_f32) return;  // a single step: read where it is used
            uint8_t *fl = fireL + (s & 1) * sp.R * HWn;
            const uint64_t key = a.fire_u8 ? 0 : a.step_seeds ? a.step_seeds[s] : a.seed;
            for (int it = kSWT - 1 - tid; it < Rw * nq; it += kSWT) {
                const int rr = it / nq, qq = it - rr * nq;
                float u[4] = {0.f, 0.f, 0.f, 0.f};
                if (!a.fire_u8) cell_uniforms4(key, (uint32_t)(a.row0 + rbase + rr), (uint32_t)(a.step0 + s), (uint32_t)qq, u);
                int cnt = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int q = 4 * qq + e, cell = rr * HWn + q;
                    if (q >= HWn) break;
                    int f;
                    if (a.fire_u8) {
                        f = a.fire_u8[((int64_t)s * a.rows + rbase + rr) * HWn + q] ? 1 : 0;
                    } else {
                        float p = a.p;
                        if (a.adaptive) {
                            int am;
                            const float cf = cell_readout(P + b * PB + ci[cell] * CP + a.out_off, 1, a.c_out, a.n_out, a.head_kind,
                                                          headL, headL + a.n_out * a.c_out, &am);
                            if (cf > a.tau || (a.given_confident && givenL[cell])) p = a.p_low;
                        }
                        f = u[e] < p ? 1 : 0;
                    }
                    fl[cell] = (uint8_t)f;
                    cnt += f;
                }
                if (cnt) atomicAdd(&firedL[rr], cnt);
            }
        };
        __syncthreads();
        if (wrap) wrap_halo(0);
        if (a.n_steps > 0) draw_fire(0, 0);
        __syncthreads();
#pragma unroll 1
        for (int s = 0; s < a.n_steps; ++s) {
            const bool more = s + 1 < a.n_steps;
#pragma unroll 1
            for (int g0 = 0; g0 < ncell; g0 += PN) {
                Pos pos = locate(g0 + sc);
                put_z(pos);
                if (g0 == 0 && more && !a.adaptive) draw_fire(s + 1, cur);
                __syncthreads();
                pass(g0, g0, s, s == 0, pos);
            }
            cur ^= 1;
            if (wrap || (a.adaptive && more)) {
                if (wrap) wrap_halo(cur);
                if (a.adaptive && more) draw_fire(s + 1, cur);
                __syncthreads();
            }
        }
        const float *Pc = P + cur * PB;
        for (int e = tid; e < Rw * C * HWn; e += kSWT) {
            const int rr = e / (C * HWn), rem = e - rr * C * HWn, c = rem / HWn, q = rem - c * HWn;
            a.x_out[rbase * C * HWn + e] = Pc[ci[rr * HWn + q] * CP + c];
        }
        if (a.conf_out) {
            float *confL = P + (cur ^ 1) * PB;  // the other buffer is free
            for (int cell = tid; cell < ncell; cell += kSWT) {
                int am;
                confL[cell] = cell_readout(Pc + ci[cell] * CP + a.out_off, 1, a.c_out, a.n_out, a.head_kind, headL,
                                           headL + a.n_out * a.c_out, &am);
            }
            __syncthreads();
            for (int rr = w; rr < Rw; rr += kSWT / 64) {
                const float sum = ordered_sum(0.0f, confL + rr * HWn, HWn);
                if (lane == 0) a.conf_out[rbase + rr] = __fdiv_rn(sum, (float)HWn);
            }
        }
        if (a.fired_out)
            for (int rr = tid; rr < Rw; rr += kSWT) a.fired_out[rbase + rr] = firedL[rr];
    }
}

}  // namespace

}  // namespace nca
