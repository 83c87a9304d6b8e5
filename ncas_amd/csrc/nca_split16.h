// fp32 cells with C = 16 channels and 128 hidden units (gfx950): the rollout of boards that fit the
// LDS in one launch (rollout_split16), and one step of boards of any size per launch
// (step_split16). In both a wave takes 16-cell tiles on its own, from the taps to the update:
// lane (cell r = lane & 15, g = lane >> 4) owns channels 4 g .. 4 g + 3 of one cell, its nine
// taps are 16-byte loads, z stays in its registers and the MLP is mlp16_split (nca_split.h) with
// the weights in LDS.
//
// Bound by the issue port: per 16-cell tile 558 VALU instructions of 4 cycles (144 of them the
// stencil, 168 the splits) and 120 MFMAs of 16, of which a SIMD overlaps little (nca_split.h). 16
// waves of up to 128 registers hide the LDS and L2 latency; 8 waves with the next tile's taps in
// registers took 110 us where these take 98. Measured (fp32 MFMA kernels before): 16 boards of
// 201x201 247 -> 98 us per step; 8 boards of 13x13 15.1 -> 6.2 us per step of a rollout in LDS; a
// single step of those 27 -> 11 us, its tiles spread over the whole device.
#pragma once

#include "nca_split.h"

namespace nca {

constexpr int kS16W = 16, kS16T = 64 * kS16W;  // waves, threads per workgroup

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void load_split16(const unsigned char *wsplit, const float *b1, unsigned char *wl, float *b1L) {
    const u32x4 *src = reinterpret_cast<const u32x4 *>(wsplit);
    u32x4 *dst = reinterpret_cast<u32x4 *>(wl);
    u32x4 v[4];
    const int n = kSplit16Frags * 64;
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = src[(int)threadIdx.x + kS16T * k < n ? threadIdx.x + kS16T * k : 0];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if ((int)threadIdx.x + kS16T * k < n) dst[threadIdx.x + kS16T * k] = v[k];
    if (threadIdx.x < 128) b1L[threadIdx.x] = b1[threadIdx.x];
}
static_assert(kSplit16Frags * 64 <= 4 * kS16T, "load_split16's rounds");

// FIRST: the first step of a call (the clamp tensor's values for the clamped channels)
template <bool IN_NCHW, bool OUT_NCHW, bool FIRST>
__global__ void __launch_bounds__(kS16T, 1) step_split16(Split16Step sp) {
    constexpr int C = 16;
    const RolloutParams &a = sp.a;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *wl = smem;
    float *b1L = reinterpret_cast<float *>(smem + kSplit16Bytes);
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, W = a.W, HWn = H * W;
    const float *kern = reinterpret_cast<const float *>(a.packed + a.off_kern);
    const float *w1 = reinterpret_cast<const float *>(a.packed + a.off_w1);
    const float *w2 = reinterpret_cast<const float *>(a.packed + a.off_w2);
    load_split16(sp.wsplit, reinterpret_cast<const float *>(a.packed + a.off_b1), wl, b1L);
    const float4 b2q = reinterpret_cast<const float4 *>(a.packed + a.off_b2)[g];
    const f32x4 b2v = {b2q.x, b2q.y, b2q.z, b2q.w};
    bool insl[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) insl[v] = 4 * g + v >= a.in_off && 4 * g + v < a.in_off + a.c_in;
    const f32x4 pq = a.padding == 1 ? reinterpret_cast<const f32x4 *>(a.packed + a.off_padv)[g] : f32x4{0.f, 0.f, 0.f, 0.f};
    const uint64_t key = a.step_seeds ? a.step_seeds[sp.step] : a.seed;
    const bool philox = !a.fire_f32 && !a.fire_u8, wrap = a.padding == 2;

    const int64_t t_begin = (int64_t)blockIdx.x * sp.tiles_per_wg;
    int64_t t_end = t_begin + sp.tiles_per_wg;
    if (t_end > sp.n_tiles) t_end = sp.n_tiles;
    const __amdgpu_buffer_rsrc_t out_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        a.x_out, (short)0, OUT_NCHW ? 0 : (int)(a.rows * HWn * C * (int64_t)sizeof(float)), 0x00020000);

    // what tile (row, tile tir of the row) loads; cells past the row's end load the last cell
    struct TileIn {
        f32x4 tp[9];
        float fin, cv[4];
        int gv, fu8, padm, qc;
    };
    auto load_tile = [&](int64_t row, int tir, TileIn &in) __attribute__((always_inline)) {
        const int q = 16 * tir + r < HWn ? 16 * tir + r : HWn - 1;
        const int i = q / W, j = q - i * W;
        in.qc = q;
        const int ro[3] = {i > 0 ? -W : (H - 1) * W, 0, i < H - 1 ? W : -(H - 1) * W};
        const int co[3] = {j > 0 ? -1 : W - 1, 0, j < W - 1 ? 1 : -(W - 1)};
        in.padm = wrap ? 0
                       : ((i == 0 ? 0x007 : 0) | (i == H - 1 ? 0x1c0 : 0) | (j == 0 ? 0x049 : 0) |
                          (j == W - 1 ? 0x124 : 0));
#pragma unroll
        for (int tt = 0; tt < 9; ++tt) {
            if (IN_NCHW) {
                const float *xr = a.x_in + (row * C + 4 * g) * (int64_t)HWn + q + ro[tt / 3] + co[tt % 3];
                in.tp[tt] = f32x4{xr[0], xr[HWn], xr[2 * HWn], xr[3 * HWn]};
            } else {
                // byte offset from the state's base, below 2^31 (checked by the host)
                const uint32_t off = ((uint32_t)(row * HWn) + (uint32_t)(q + ro[tt / 3] + co[tt % 3])) * (uint32_t)(4 * C) +
                                     16u * (uint32_t)g;
                in.tp[tt] = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const unsigned char *>(a.x_in) + off);
            }
        }
        const int64_t cell = row * HWn + q;
        in.gv = a.given[cell];
        // loaded without a branch (an absent mask loads something else, unused)
        in.fin = *(a.fire_f32 ? a.fire_f32 + cell : a.x_in + cell);
        in.fu8 = *(a.fire_u8 ? a.fire_u8 + cell : a.given + cell);
        if (FIRST) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int ci = insl[v] ? 4 * g + v - a.in_off : 0;
                in.cv[v] = a.c_in > 0 ? a.clamp[(row * a.c_in + ci) * (int64_t)HWn + q] : 0.0f;
            }
        }
    };

    int64_t cur_row = -1;
    int fired_run = 0;
    auto flush_fired = [&]() {
        int s = fired_run;
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o);
        if (lane == 0 && s && a.fired_out) atomicAdd(a.fired_out + cur_row, s);
        fired_run = 0;
    };
    // Philox for 16 of the wave's tiles at a time: lane L evaluates cell quad L & 3 of the tile L >> 2
    // tiles ahead and keeps the four uniforms; tile k's cell r reads lane 4 k + r / 4's word r % 4
    float u4[4] = {0.f, 0.f, 0.f, 0.f};
    int kgrp = 0;
    const int tpr = sp.tiles_per_row;
    auto draw16 = [&](int64_t row, int tir) {
        int ti = tir + kS16W * (lane >> 2);
        int64_t rw = row;
        while (ti >= tpr) {
            ti -= tpr;
            ++rw;
        }
        cell_uniforms4(key, (uint32_t)(a.row0 + rw), (uint32_t)(a.step0 + sp.step), (uint32_t)(4 * ti + (lane & 3)), u4);
    };

    auto process = [&](TileIn &in, int64_t row, int tir) __attribute__((always_inline)) {
        const int q = 16 * tir + r;
        const bool valid = q < HWn;
        if (__ballot(in.padm != 0)) {  // tiles with a cell on the grid's edge (the centre tap never is one)
#pragma unroll
            for (int tt = 0; tt < 9; ++tt) {
                if (tt == 4) continue;
                const bool p = (in.padm >> tt) & 1;
#pragma unroll
                for (int c = 0; c < 4; ++c) in.tp[tt][c] = p ? pq[c] : in.tp[tt][c];
            }
        }
        float z[4][4];
        stencil16(in.tp, kern, z);
        const f32x4 dx = mlp16_split(z, wl, b1L, b2v, w1, w2, lane);
        float f;
        if (philox) {
            const int src = 4 * kgrp + (r >> 2);
            const float a0 = __shfl(u4[0], src), a1 = __shfl(u4[1], src), a2 = __shfl(u4[2], src), a3 = __shfl(u4[3], src);
            const float u = (r & 3) == 0 ? a0 : (r & 3) == 1 ? a1 : (r & 3) == 2 ? a2 : a3;
            float p = a.p;
            if (a.adaptive) {
                const float *hw = reinterpret_cast<const float *>(a.packed + a.off_headw);
                const float *hb = reinterpret_cast<const float *>(a.packed + a.off_headb);
                int am;
                const float *xc = IN_NCHW ? a.x_in + (row * C + a.out_off) * (int64_t)HWn + in.qc
                                          : a.x_in + (row * HWn + in.qc) * C + a.out_off;
                const float cf = cell_readout(xc, IN_NCHW ? HWn : 1, a.c_out, a.n_out, a.head_kind, hw, hb, &am);
                if (cf > a.tau || (a.given_confident && in.gv)) p = a.p_low;
            }
            f = u < p ? 1.0f : 0.0f;
        } else {
            f = a.fire_f32 ? in.fin : in.fu8 ? 1.0f : 0.0f;
        }
        const bool gv = in.gv != 0;
        const f32x4 xo = in.tp[4];
        f32x4 u;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            float uv = __fadd_rn(xo[v], __fmul_rn(f, dx[v]));
            if (a.noise) uv = __fadd_rn(uv, a.noise[(row * C + 4 * g + v) * (int64_t)HWn + in.qc]);
            u[v] = (gv && insl[v]) ? (FIRST ? in.cv[v] : xo[v]) : uv;
        }
        if (OUT_NCHW) {
            if (valid) {
                float *xr = a.x_out + (row * C + 4 * g) * (int64_t)HWn + q;
#pragma unroll
                for (int v = 0; v < 4; ++v) xr[(int64_t)v * HWn] = u[v];
            }
        } else {
            // cells past the row's end store beyond the buffer, which the hardware drops
            const uint32_t off = valid ? ((uint32_t)(row * HWn + q) * (uint32_t)C + 4u * (uint32_t)g) * 4u : 0x80000000u;
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, u), out_rsrc, off, 0, 0);
        }
        if (a.fired_out) fired_run += (valid && g == 0 && f != 0.0f) ? 1 : 0;
    };

    int64_t t = t_begin + w;
    int64_t row = t / tpr;
    int tir = (int)(t - row * tpr);
    __syncthreads();  // the weights
    for (; t < t_end; t += kS16W) {
        asm volatile("" ::: "memory");  // the weights' LDS reads stay in the loop (240 registers otherwise)
        TileIn in;
        load_tile(row, tir, in);
        if (a.fired_out && row != cur_row) {
            if (cur_row >= 0) flush_fired();
            cur_row = row;
        }
        if (philox && kgrp == 0) draw16(row, tir);
        process(in, row, tir);
        kgrp = (kgrp + 1) & 15;
        tir += kS16W;
        while (tir >= tpr) {
            tir -= tpr;
            ++row;
        }
    }
    if (a.fired_out && cur_row >= 0) flush_fired();
}

// R rows' whole rollout in LDS: the state twice (the step reads one, writes the other), cells of 64
// bytes with a one-cell border; the tiles of all rows' cells go round the 16 waves; one barrier
// per step (a second with wrap padding, whose border is copied, or gated firing, which reads the
// new state). The fire bytes of the next step are drawn beside this one's tiles by the waves with
// the fewest.
__global__ void __launch_bounds__(kS16T, 1) rollout_split16(Split16Resident sp) {
    constexpr int C = 16;
    const RolloutParams &a = sp.a;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *wl = smem;
    float *b1L = reinterpret_cast<float *>(smem + kSplit16Bytes);
    float *P = reinterpret_cast<float *>(smem + sp.l_P);
    uint16_t *ci = reinterpret_cast<uint16_t *>(smem + sp.l_ci);  // cell -> bordered cell
    uint8_t *fireL = smem + sp.l_fire, *givenL = smem + sp.l_given;
    int *firedL = reinterpret_cast<int *>(smem + sp.l_fired);
    float *headL = reinterpret_cast<float *>(smem + sp.l_head);
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, W = a.W, HWn = H * W, Wp = W + 2, HWp = (H + 2) * Wp;
    const int64_t rbase = (int64_t)blockIdx.x * sp.R;
    const int Rw = (int)(a.rows - rbase < sp.R ? a.rows - rbase : sp.R);
    const int ncell = Rw * HWn, ntile = (ncell + 15) >> 4, PB = sp.R * HWp * C;  // floats per buffer
    const float *kern = reinterpret_cast<const float *>(a.packed + a.off_kern);
    const float *w1 = reinterpret_cast<const float *>(a.packed + a.off_w1);
    const float *w2 = reinterpret_cast<const float *>(a.packed + a.off_w2);
    load_split16(sp.wsplit, reinterpret_cast<const float *>(a.packed + a.off_b1), wl, b1L);
    const float4 b2q = reinterpret_cast<const float4 *>(a.packed + a.off_b2)[g];
    const f32x4 b2v = {b2q.x, b2q.y, b2q.z, b2q.w};
    bool insl[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) insl[v] = 4 * g + v >= a.in_off && 4 * g + v < a.in_off + a.c_in;
    // ---- the rows' state, given flags and cell table; the constant border
    for (int e = tid; e < Rw * C * HWn; e += kS16T) {
        const int rr = e / (C * HWn), rem = e - rr * C * HWn, c = rem / HWn, q = rem - c * HWn;
        const float v = a.x_in[rbase * C * HWn + e];
        P[(rr * HWp + (q / W + 1) * Wp + q % W + 1) * C + c] = v;
        if (a.x_rec0) a.x_rec0[rbase * C * HWn + e] = v;
    }
    for (int e = tid; e < ncell; e += kS16T) {
        const int rr = e / HWn, q = e - rr * HWn;
        givenL[e] = a.given[rbase * HWn + e];
        ci[e] = (uint16_t)(rr * HWp + (q / W + 1) * Wp + q % W + 1);
    }
    for (int e = tid; e < sp.R; e += kS16T) firedL[e] = 0;
    {
        const float *hw = reinterpret_cast<const float *>(a.packed + a.off_headw);
        const float *hb = reinterpret_cast<const float *>(a.packed + a.off_headb);
        const int nw = a.n_out * a.c_out;
        for (int e = tid; e < nw + a.n_out; e += kS16T) headL[e] = e < nw ? hw[e] : hb[e - nw];
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
    if (a.padding != 2) {
        const float *padv = reinterpret_cast<const float *>(a.packed + a.off_padv);
        for (int e = tid; e < 2 * Rw * nhalo * C; e += kS16T) {
            const int c = e % C, rest = e / C, h = rest % nhalo, rb = rest / nhalo, rr = rb % Rw, buf = rb / Rw;
            int ip, jp;
            halo_cell(h, ip, jp);
            P[buf * PB + (rr * HWp + ip * Wp + jp) * C + c] = a.padding == 1 ? padv[c] : 0.0f;
        }
    }
    auto wrap_halo = [&](int buf) {
        for (int e = tid; e < Rw * nhalo * 4; e += kS16T) {
            const int qd = e & 3, rest = e >> 2, h = rest % nhalo, rr = rest / nhalo;
            int ip, jp;
            halo_cell(h, ip, jp);
            const int si = ip == 0 ? H : ip == H + 1 ? 1 : ip, sj = jp == 0 ? W : jp == W + 1 ? 1 : jp;
            float *p = P + buf * PB + rr * HWp * C + 4 * qd;
            *reinterpret_cast<float4 *>(p + (ip * Wp + jp) * C) = *reinterpret_cast<const float4 *>(p + (si * Wp + sj) * C);
        }
    };
    // fire bytes of step s (the state in buffer cur is the step's input) into half s & 1
    const int nq = (HWn + 3) >> 2;
    const bool from_mask = a.fire_u8 != nullptr;
    auto draw_fire = [&](int s, int cur) {
        if (a.fire_f32) return;  // a single step: read where it is used
        uint8_t *fl = fireL + (s & 1) * sp.R * HWn;
        const uint64_t key = from_mask ? 0 : a.step_seeds ? a.step_seeds[s] : a.seed;
        for (int it = kS16T - 1 - tid; it < Rw * nq; it += kS16T) {
            const int rr = it / nq, qq = it - rr * nq;
            float u[4] = {0.f, 0.f, 0.f, 0.f};
            if (!from_mask) cell_uniforms4(key, (uint32_t)(a.row0 + rbase + rr), (uint32_t)(a.step0 + s), (uint32_t)qq, u);
            int cnt = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int q = 4 * qq + e, cell = rr * HWn + q;
                if (q >= HWn) break;
                int f;
                if (from_mask) {
                    f = a.fire_u8[((int64_t)s * a.rows + rbase + rr) * HWn + q] ? 1 : 0;
                } else {
                    float p = a.p;
                    if (a.adaptive) {
                        int am;
                        const float cf = cell_readout(P + cur * PB + ci[cell] * C + a.out_off, 1, a.c_out, a.n_out, a.head_kind,
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
    if (a.padding == 2) wrap_halo(0);
    if (a.n_steps > 0) draw_fire(0, 0);
    __syncthreads();
    int toff[9];  // floats
#pragma unroll
    for (int t9 = 0; t9 < 9; ++t9) toff[t9] = ((t9 / 3 - 1) * Wp + t9 % 3 - 1) * C;

    int cur = 0;
    for (int s = 0; s < a.n_steps; ++s) {
        const uint8_t *fl = fireL + (s & 1) * sp.R * HWn;
        const float *Pc = P + cur * PB;
        float *Pn = P + (cur ^ 1) * PB;
        for (int t = w; t < ntile; t += kS16W) {
            const int gq = 16 * t + r, gc = gq < ncell ? gq : ncell - 1;
            const int pc = ci[gc] * C + 4 * g;
            f32x4 tp[9];
#pragma unroll
            for (int t9 = 0; t9 < 9; ++t9) tp[t9] = *reinterpret_cast<const f32x4 *>(Pc + pc + toff[t9]);
            const bool gv = givenL[gc] != 0;
            float f = fl[gc] ? 1.0f : 0.0f;
            float z[4][4];
            stencil16(tp, kern, z);
            const f32x4 dx = mlp16_split(z, wl, b1L, b2v, w1, w2, lane);
            const f32x4 xo = tp[4];
            const int rr = gc / HWn, q = gc - rr * HWn;
            const int64_t row = rbase + rr;
            if (a.fire_f32) {
                f = a.fire_f32[row * HWn + q];
                if (gq < ncell && g == 0 && f != 0.0f) atomicAdd(&firedL[rr], 1);
            }
            f32x4 u;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int c = 4 * g + v;
                float uv = __fadd_rn(xo[v], __fmul_rn(f, dx[v]));
                if (a.noise) uv = __fadd_rn(uv, a.noise[(row * C + c) * (int64_t)HWn + q]);
                u[v] = (gv && insl[v]) ? (s == 0 ? a.clamp[(row * a.c_in + c - a.in_off) * (int64_t)HWn + q] : xo[v]) : uv;
            }
            if (gq < ncell) {
                *reinterpret_cast<f32x4 *>(Pn + pc) = u;
                if (a.x_rec) {
                    float *xr = a.x_rec + s * a.rec_stride + (row * C + 4 * g) * (int64_t)HWn + q;
#pragma unroll
                    for (int v = 0; v < 4; ++v) xr[(int64_t)v * HWn] = u[v];
                }
            }
        }
        const bool more = s + 1 < a.n_steps;
        if (more && !a.adaptive) draw_fire(s + 1, cur);
        __syncthreads();
        cur ^= 1;
        if (a.padding == 2 || (a.adaptive && more)) {
            if (a.padding == 2) wrap_halo(cur);
            if (a.adaptive && more) draw_fire(s + 1, cur);
            __syncthreads();
        }
    }
    const float *Pc = P + cur * PB;
    for (int e = tid; e < Rw * C * HWn; e += kS16T) {
        const int rr = e / (C * HWn), rem = e - rr * C * HWn, c = rem / HWn, q = rem - c * HWn;
        a.x_out[rbase * C * HWn + e] = Pc[ci[rr * HWn + q] * C + c];
    }
    if (a.conf_out) {
        float *confL = P + (cur ^ 1) * PB;  // the other buffer is free
        for (int cell = tid; cell < ncell; cell += kS16T) {
            int am;
            confL[cell] = cell_readout(Pc + ci[cell] * C + a.out_off, 1, a.c_out, a.n_out, a.head_kind, headL,
                                       headL + a.n_out * a.c_out, &am);
        }
        __syncthreads();
        for (int rr = w; rr < Rw; rr += kS16W) {
            const float sum = ordered_sum(0.0f, confL + rr * HWn, HWn);
            if (lane == 0) a.conf_out[rbase + rr] = __fdiv_rn(sum, (float)HWn);
        }
    }
    if (a.fired_out)
        for (int rr = tid; rr < Rw; rr += kS16T) a.fired_out[rbase + rr] = firedL[rr];
}

}  // namespace

}  // namespace nca
