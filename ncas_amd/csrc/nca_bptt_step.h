// One step of the BPTT backward in one launch, for every cell that mlp_back32 does not take (C = 16
// and 64 in both precisions, C = 32 in fp32), and the weight gradients of several steps in one
// more.
//
// `back_step`: a workgroup of 4 waves owns tiles of 32 consecutive cells (m = row * HW + q). For a
// tile it
//   1. finishes the gradient of the step's output state: the later step's g_u plus the transposed
//      stencil of its g_z (of this cell's neighbours, written by the previous launch), the loss
//      head's gradient, the clamp's and the fire mask's backward -> g_u, g_dx;
//   2. recomputes z from the step's input state (9 taps, 4 kernels);
//   3. on MFMA, wave w for a quarter of the hidden units: h = relu(W1 z + b1), g_a = (W2^T g_dx)
//      [h > 0]; then for a quarter of the features g_z = W1^T g_a;
//   4. adds the kernel-weight, head and loss sums of its cells into its own slots.
// Only g_z crosses workgroups, and only from one launch to the next, so a step is one launch. It is
// bound by latency at training sizes (10,368 cells of 9x9 are 324 tiles for 256 CUs): the weight
// fragments come from the L2 once per tile, 16 bytes a lane, instead of staying in registers, so
// that two workgroups fit a CU and the fp32 C = 64 cell (576 KB of weights) runs the same code.
//
// z, h, g_a and g_dx of up to G steps (160 MB) are kept tile-major ([tile][feature][32 cells]: a tile's
// stores are one contiguous run, and so are 16 features of 32 cells, an MFMA operand), and
// `weight_grads` sums dW1 = g_a z^T, dW2 = g_dx h^T, db1 and db2 over all their cells at once: a
// split-K product over G * M cells writes its partial sums once per group where one over each
// step's M cells read and wrote all of them every step (84 MB a step for C = 64).
//
// Against the five GEMM launches, row sums, front, stencil and strip kernels that did a step
// before (128 boards of 9x9, C = 64, bf16, 32 steps: 665 -> 46 us a step and 62 us per group of 9
// steps; 64 boards of 13x13, C = 16, fp32: 117 -> 22 us a step and 70 us per group of 11). Every
// stage issues its loads before it uses the first (one at a time they took twice as long: the
// compiler packs each pair of taps as it arrives), the weight fragments' loads are in flight
// beside the head, the stores come last (a load waits for the stores issued before it), and the
// LDS plan lets two workgroups share a CU (with one the 324 tiles take two rounds: 66 us).
#pragma once

#include <type_traits>

#include "nca_device.h"

namespace {

constexpr int kBN = 32;            // cells per tile of back_step
constexpr int kBackMaxWgs = 512;   // workgroups of back_step (two per CU), each with slots of its own
constexpr int kGroupSplits = 256;  // most K ranges (slots) of weight_grads

template <int C, int HD, bool BF16>
struct BShape {
    static constexpr int F = 4 * C;
    static constexpr int ES = BF16 ? 2 : 4;     // bytes per element of z, h, g_a, g_dx, g_z
    static constexpr int EB = 16 / ES;          // elements in a lane's 16 bytes
    static constexpr int KB = 4 * EB;           // k per fragment block (16 rows x KB)
    static constexpr int KF = F / KB;           // blocks of fc1's k axis
    static constexpr int KC = (C + KB - 1) / KB;  // of W2^T's (zero-padded for bf16 C = 16)
    static constexpr int KH = HD / KB;          // of W1^T's
    static constexpr int MT1 = HD / 64;         // hidden m-tiles per wave
    static constexpr int MT2 = F / 64;          // feature m-tiles per wave
    static constexpr int ZS = F + EB, GS = HD + EB, DS = KC * KB + EB;  // LDS row strides (elements)
    static constexpr int NZ = kBN * (C / 4) / 256 > 0 ? kBN * (C / 4) / 256 : 1;  // items per thread
    static constexpr int ITEMS = kBN * (C / 4);
    // fp32 h goes straight to its kept buffer (64-byte runs): with it in LDS only one workgroup of the
    // C = 32 cell would fit a CU
    static constexpr unsigned Z = 0, H = Z + kBN * ZS * ES, GA = H + (BF16 ? kBN * GS * ES : 0), GZ = GA + kBN * GS * ES,
                              GD = GZ + kBN * ZS * ES, END = GD + kBN * DS * ES;
    // LDS column of MFMA operand row element k: a lane reads its 16 bytes of a block at 16 g. fp32: lane
    // group g's element j is k = 4 j + g of the 16, so that the k axis is summed in ascending fours
    static __device__ __forceinline__ int col(int k) { return BF16 ? k : (k & ~15) | ((k & 3) << 2) | ((k >> 2) & 3); }
};

// Fragment images in the packed weights (nca_layout.h): [m-tile][k-block][lane] 16-byte units.
template <bool BF16>
struct BFrag;
template <>
struct BFrag<true> {
    typedef nca::bf16x8 type;
    static __device__ __forceinline__ nca::f32x4 mma(type a, type b, nca::f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <>
struct BFrag<false> {
    typedef nca::f32x4 type;
    // slot j of lane group g is k = 4 j + g in both operands
    static __device__ __forceinline__ nca::f32x4 mma(type a, type b, nca::f32x4 c) {
#pragma unroll
        for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
        return c;
    }
};

template <bool BF16>
__device__ __forceinline__ void put4(unsigned char *p, const float v[4]) {
    if (BF16)
        *reinterpret_cast<uint2 *>(p) = make_uint2(nca::pack_bf16x2(v[0], v[1]), nca::pack_bf16x2(v[2], v[3]));
    else
        *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
template <bool BF16>
__device__ __forceinline__ void get4(const unsigned char *p, float v[4]) {
    if (BF16) {
        const uint2 u = *reinterpret_cast<const uint2 *>(p);
        v[0] = nca::bf16_lo(u.x), v[1] = nca::bf16_hi(u.x), v[2] = nca::bf16_lo(u.y), v[3] = nca::bf16_hi(u.y);
    } else {
        const float4 u = *reinterpret_cast<const float4 *>(p);
        v[0] = u.x, v[1] = u.y, v[2] = u.z, v[3] = u.w;
    }
}
template <bool BF16>
__device__ __forceinline__ float rnd(float v) { return BF16 ? nca::round_bf16(v) : v; }

struct BackStepArgs {
    FrontArgs f;             // x1, gin (NCHW, the chunk's last step only), targets, masks, head; Gu: (M, C)
    const float *xt;         // the step's input state (rows, C, H, W)
    const void *gz_in;       // g_z of the later step (M, F), or null
    void *gz_out;            // (M, F)
    const uint4 *w1, *w1t, *w2t;
    const float *b1, *kern, *padv;
    void *zs, *hs, *gas, *gds;  // kept buffers, [tile][feature][32 cells], this step's tiles from tile0
    int64_t tile0;
    float *slots;            // (workgroups, nslot): dK (36), dhead, head bias, loss
    int nslot, accum;        // accum: add to the slots' contents
    int64_t tiles;
    uint32_t *status;        // the workspace's backward status word, cleared by the first launch
};

// A wave's weight fragments of one product: MT m-tiles, K k-blocks, of which up to PRE are in
// registers: `load` issues the first ones (early, so that their latency passes beside other work),
// `mma` adds A B to acc (B rows from LDS) and refills each slot once it is used.
template <bool BF16, int MT, int K>
struct WFrags {
    typedef typename BFrag<BF16>::type fr;
    static constexpr int PRE = K < (BF16 ? 8 : 4) ? K : (BF16 ? 8 : 4);
    const uint4 *base;  // uniform
    uint4 f[PRE][MT];
    __device__ __forceinline__ uint4 at(int m, int k, int lane) const { return (base + (m * K + k) * 64)[lane]; }
    __device__ __forceinline__ void load(const uint4 *img, int mt0, int lane) {
        base = img + (int64_t)mt0 * K * 64;
#pragma unroll
        for (int k = 0; k < PRE; ++k)
#pragma unroll
            for (int m = 0; m < MT; ++m) f[k][m] = at(m, k, lane);
    }
    __device__ __forceinline__ void mma(const unsigned char *b, int stride_bytes, int lane, nca::f32x4 (&acc)[MT][2]) {
        const unsigned char *br = b + (lane & 15) * stride_bytes + 16 * (lane >> 4);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            __builtin_amdgcn_sched_barrier(0);
            fr bv[2];
#pragma unroll
            for (int n = 0; n < 2; ++n) bv[n] = *reinterpret_cast<const fr *>(br + 16 * n * stride_bytes + 64 * k);
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n) acc[m][n] = BFrag<BF16>::mma(__builtin_bit_cast(fr, f[k % PRE][m]), bv[n], acc[m][n]);
            if (k + PRE < K) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = 0; m < MT; ++m) f[k % PRE][m] = at(m, k + PRE, lane);
            }
        }
    }
};

// The gradient reaching cell (i, j) of board row `row`, channels [c0, c0 + 4), from the later step:
// its g_u plus the transposed stencil of its g_z (M, F). The loads
// (of 9 neighbours, or of a row of 3 in fp32) are issued before their sums; a neighbour beyond a wall or zero border contributes nothing.
template <int C, bool BF16>
__device__ __forceinline__ void later_grad(const Dims &d, const float *Gu, const void *Gz, const float *kern, int64_t mrow,
                                           int i, int j, int c0, float g[4]) {
    constexpr int F = 4 * C, ES = BF16 ? 2 : 4;
    typedef std::conditional_t<BF16, uint2, float4> raw_t;
    const unsigned char *gz = static_cast<const unsigned char *>(Gz);
    const float4 g4 = *reinterpret_cast<const float4 *>(Gu + (mrow + i * d.W + j) * C + c0);
    constexpr int R = BF16 ? 9 : 3;  // neighbours at a time
    g[0] = g4.x, g[1] = g4.y, g[2] = g4.z, g[3] = g4.w;
#pragma unroll
    for (int t0 = 0; t0 < 9; t0 += R) {
        raw_t v[R][4];
        unsigned in = 0;
#pragma unroll
        for (int t = 0; t < R; ++t) {
            // the cell whose tap t0 + t reads this cell
            const int q = neighbour(i, j, 1 - (t0 + t) / 3, 1 - (t0 + t) % 3, d.H, d.W, d.padding);
            in |= (q >= 0 ? 1u : 0u) << t;
            const unsigned char *p = gz + ((mrow + (q < 0 ? 0 : q)) * F + c0) * ES;
#pragma unroll
            for (int k = 0; k < 4; ++k) v[t][k] = *reinterpret_cast<const raw_t *>(p + k * C * ES);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const bool ok = (in >> t) & 1u;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float f[4];
                get4<BF16>(reinterpret_cast<const unsigned char *>(&v[t][k]), f);
                const float w = kern[k * 9 + t0 + t];
#pragma unroll
                for (int c = 0; c < 4; ++c) g[c] = ok ? __builtin_fmaf(w, f[c], g[c]) : g[c];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The 9 taps of channels [c0, c0 + 4) of cell (i, j) of a board row (rounded to bf16 for bf16 cells).
template <int C, bool BF16>
__device__ __forceinline__ void cell_taps(const Dims &d, const float *xt, const float *padv, int row, int i, int j, int c0,
                                          float xv[4][9]) {
    const float *xr = xt + ((int64_t)row * C + c0) * d.HW;
    float hv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (d.padding == 1) {
#pragma unroll
        for (int c = 0; c < 4; ++c) hv[c] = padv[c0 + c];
    }
    unsigned in = 0;
#pragma unroll
    for (int t = 0; t < 9; ++t) {
        const int nq = neighbour(i, j, t / 3 - 1, t % 3 - 1, d.H, d.W, d.padding);
        in |= (nq >= 0 ? 1u : 0u) << t;
        const float *xp = xr + (nq < 0 ? 0 : nq);
#pragma unroll
        for (int c = 0; c < 4; ++c) xv[c][t] = xp[c * d.HW];
    }
    __builtin_amdgcn_sched_barrier(0);  // every load issued before the first use
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int c = 0; c < 4; ++c) xv[c][t] = rnd<BF16>((in >> t) & 1u ? xv[c][t] : hv[c]);
}

// A tile's LDS rows (cells) out to a kept buffer, transposed to (feats, 32 cells), 16 bytes a lane.
template <class S, bool BF16, bool PERM>
__device__ __forceinline__ void flush_tile(const unsigned char *L, int stride, int feats, void *out, int64_t tile) {
    constexpr int PARTS = kBN / S::EB;
    uint4 *o = static_cast<uint4 *>(out) + tile * feats * PARTS;
    for (int e = threadIdx.x; e < feats * PARTS; e += 256) {
        const int part = e % PARTS, f = e / PARTS;
        const unsigned char *src = L + (part * S::EB * stride + (PERM ? S::col(f) : f)) * S::ES;
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            w[i] = BF16 ? *reinterpret_cast<const uint16_t *>(src + 2 * i * stride * 2) |
                              ((uint32_t)*reinterpret_cast<const uint16_t *>(src + (2 * i + 1) * stride * 2) << 16)
                        : *reinterpret_cast<const uint32_t *>(src + i * stride * 4);
        o[e] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

template <int C, int HD, bool BF16, int NO>
__global__ void __launch_bounds__(256, 2) back_step(BackStepArgs a) {
    using S = BShape<C, HD, BF16>;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // the head: weights [v][c] and transposed [c][v], bias; per cell: logit gradients, output channels
    __shared__ __attribute__((aligned(16))) float hwL[NO * NO], hwT[NO][NO], hbL[NO];
    __shared__ float mxL[kBN], fireL[kBN], lossL[kBN], mkL[kBN], red[16 * 36];
    __shared__ int givenL[kBN], rowL[kBN], iL[kBN], jL[kBN], tgtL[kBN];
    // the head's per-cell values are done with before g_a and g_z are written: they share their LDS
    // (so that two workgroups of the bf16 C = 64 cell fit a CU)
    struct Head {
        float gl[kBN][NO], xo[kBN][NO], lg[kBN][NO + 1], ex[kBN][NO + 1];
    };
    static_assert(sizeof(Head) <= S::GD - S::GA, "the head's values exceed g_a's and g_z's LDS");
    Head &hd = *reinterpret_cast<Head *>(smem + S::GA);
    auto &glL = hd.gl, &xoL = hd.xo;
    auto &lgL = hd.lg, &exL = hd.ex;
    unsigned char *ZL = smem + S::Z, *HL = smem + S::H, *GAL = smem + S::GA, *GZL = smem + S::GZ, *GDL = smem + S::GD;
    const Dims &d = a.f.d;
    int tid = threadIdx.x;
    const bool has_loss = a.f.wscale != 0.0f;
    const int M = (int)d.M;
    if (has_loss) {
        for (int i = tid; i < NO * NO; i += 256) {
            const int v = i / NO, c = i - v * NO;
            const float w = v < d.n_out && c < d.c_out ? a.f.head_w[v * d.c_out + c] : 0.0f;
            hwL[i] = w;
            hwT[c][v] = w;
        }
        if (tid < NO) hbL[tid] = tid < d.n_out ? a.f.head_b[tid] : 0.0f;
    }
    if (S::KC * S::KB > C)  // the zero part of g_dx's k axis
        for (int i = tid; i < kBN * S::DS; i += 256) reinterpret_cast<uint16_t *>(GDL)[i] = 0;
    for (int i = tid; i < 16 * 36; i += 256) red[i] = 0.0f;
    if (!a.accum && blockIdx.x == 0 && tid == 0) *a.status = 0;
    const int npw = d.n_out * d.c_out, np = npw + d.n_out;
    float hs[2] = {0.0f, 0.0f}, lossv = 0.0f;
    const float denom = has_loss && a.f.mask ? *a.f.denom : 1.0f;

    for (int64_t tile = blockIdx.x; tile < a.tiles; tile += gridDim.x) {
        // opaque per tile: the address arithmetic stays in the loop (hoisted out of it, it spills)
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, g = lane >> 4, l16 = lane & 15;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: the fragments' addresses are scalar
        const int m0 = (int)(tile * kBN);
        if (tid < kBN) {
            const int m = m0 + tid < M ? m0 + tid : M - 1, row = m / d.HW, q = m - row * d.HW, i = q / d.W;
            rowL[tid] = row;
            iL[tid] = i;
            jL[tid] = q - i * d.W;
        }
        __syncthreads();
        // ---- per cell (wave 3): given flag and fire value; the head's output channels
        if (has_loss) {
#pragma unroll
            for (int it = 0; it < (kBN * NO + 255) / 256; ++it) {
                const int e = tid + 256 * it;
                if (e >= kBN * NO) continue;
                const int n = e & (kBN - 1), c = e / kBN;
                const int q = iL[n] * d.W + jL[n];
                xoL[n][c] = c < d.c_out ? a.f.x1[((int64_t)rowL[n] * C + d.out_off + c) * d.HW + q] : 0.0f;
            }
        }
        if (tid >= 192 && tid < 192 + kBN) {
            const int n = tid - 192, m = m0 + n;
            float f = 0.0f;
            int gv = 0;
            if (m < M) {
                gv = a.f.given[m] != 0;
                if (a.f.fire_f32) {
                    f = a.f.fire_f32[m];
                } else if (a.f.fire_u8) {
                    f = a.f.fire_u8[m] ? 1.0f : 0.0f;
                } else {
                    const int q = iL[n] * d.W + jL[n], e4 = q & 3;
                    float u[4];
                    nca::cell_uniforms4(a.f.key_ptr ? *a.f.key_ptr : a.f.key, (uint32_t)(a.f.row0 + rowL[n]), a.f.step,
                                        (uint32_t)(q >> 2), u);
                    f = (e4 == 0 ? u[0] : e4 == 1 ? u[1] : e4 == 2 ? u[2] : u[3]) < a.f.p ? 1.0f : 0.0f;
                }
            }
            fireL[n] = f;
            givenL[n] = gv;
            tgtL[n] = has_loss && m < M ? a.f.targets[m] : 0;
            mkL[n] = has_loss && a.f.mask && m < M ? a.f.mask[m] : 0.0f;
        }
        // ---- z: item (cell n, channel quad), lanes over cells
#pragma unroll
        for (int it = 0; it < S::NZ; ++it) {
            const int e = tid + 256 * it, n = e & (kBN - 1), c0 = 4 * (e / kBN);
            if (e >= S::ITEMS) continue;
            const bool ok = m0 + n < M;
            float xv[4][9];
            cell_taps<C, BF16>(d, a.xt, a.padv, rowL[n], iL[n], jL[n], c0, xv);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float z[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    float s = 0.0f;
#pragma unroll
                    for (int t = 0; t < 9; ++t) s = __builtin_fmaf(a.kern[k * 9 + t], xv[c][t], s);
                    z[c] = ok ? rnd<BF16>(s) : 0.0f;
                }
                if (BF16) {
                    put4<BF16>(ZL + (n * S::ZS + k * C + c0) * S::ES, z);
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c) reinterpret_cast<float *>(ZL)[n * S::ZS + S::col(k * C + c0 + c)] = z[c];
                }
            }
        }
        // ---- the gradient of the output state: item (cell n, channel quad), lanes over quads
        float gg[S::NZ][4];
#pragma unroll
        for (int it = 0; it < S::NZ; ++it) {
            const int e = tid + 256 * it, c0 = 4 * (e & (C / 4 - 1)), n = e / (C / 4);
#pragma unroll
            for (int c = 0; c < 4; ++c) gg[it][c] = 0.0f;
            if (e >= S::ITEMS || m0 + n >= M) continue;
            const int row = rowL[n], i = iL[n], j = jL[n];
            if (a.gz_in) {
                later_grad<C, BF16>(d, a.f.Gu, a.gz_in, a.kern, (int64_t)row * d.HW, i, j, c0, gg[it]);
            } else if (a.f.gin) {
#pragma unroll
                for (int c = 0; c < 4; ++c) gg[it][c] = a.f.gin[((int64_t)row * C + c0 + c) * d.HW + i * d.W + j];
            }
        }
        __syncthreads();
        WFrags<BF16, S::MT1, S::KF> w1;
        WFrags<BF16, S::MT1, S::KC> w2t;
        w1.load(a.w1, wave * S::MT1, lane);
        w2t.load(a.w2t, wave * S::MT1, lane);
        // ---- the loss head, thread (cell, class): the logit, its exponential, the soft-max gradient
        if (has_loss) {
#pragma unroll
            for (int it = 0; it < (kBN * NO + 255) / 256; ++it) {
                const int e = tid + 256 * it;
                if (e >= kBN * NO) continue;
                const int n = e & (kBN - 1), v = e / kBN;
                float acc = hbL[v];
#pragma unroll
                for (int c = 0; c < NO; ++c) acc = c < d.c_out ? __builtin_fmaf(hwL[v * NO + c], xoL[n][c], acc) : acc;
                lgL[n][v] = acc;
            }
            __syncthreads();
#pragma unroll
            for (int it = 0; it < (kBN * NO + 255) / 256; ++it) {
                const int e = tid + 256 * it;
                if (e >= kBN * NO) continue;
                const int n = e & (kBN - 1), v = e / kBN;
                float mx = -INFINITY;
#pragma unroll
                for (int w = 0; w < NO; ++w) mx = w < d.n_out ? fmaxf(mx, lgL[n][w]) : mx;
                exL[n][v] = v < d.n_out ? expf(lgL[n][v] - mx) : 0.0f;
                if (v == 0) mxL[n] = mx;
            }
            __syncthreads();
#pragma unroll
            for (int it = 0; it < (kBN * NO + 255) / 256; ++it) {
                const int e = tid + 256 * it;
                if (e >= kBN * NO) continue;
                const int n = e & (kBN - 1), v = e / kBN, tgt = tgtL[n];
                const float scale = a.f.mask ? a.f.wscale * mkL[n] / denom : a.f.wscale;
                float s = 0.0f;
#pragma unroll
                for (int w = 0; w < NO; ++w) s += exL[n][w];
                const bool ok = m0 + n < M;
                glL[n][v] = ok && v < d.n_out ? (exL[n][v] / s - (v == tgt ? 1.0f : 0.0f)) * scale : 0.0f;
                if (v == 0)
                    lossL[n] = ok ? (mxL[n] + logf(s) - (tgt >= 0 && tgt < d.n_out ? lgL[n][tgt] : mxL[n])) * scale : 0.0f;
            }
            __syncthreads();
        }
        // ---- clamp and fire: g_u, g_dx
#pragma unroll
        for (int it = 0; it < S::NZ; ++it) {
            const int e = tid + 256 * it, c0 = 4 * (e & (C / 4 - 1)), n = e / (C / 4);
            if (e >= S::ITEMS) continue;
            const bool gv = givenL[n] != 0, ok = m0 + n < M;
            const float f = fireL[n];
            float gd[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int ch = c0 + c, co = ch - d.out_off;
                float v = gg[it][c];
                if (has_loss && co >= 0 && co < d.c_out) {
#pragma unroll
                    for (int o = 0; o < NO; ++o) v = __builtin_fmaf(hwT[co][o], glL[n][o], v);
                }
                if (gv && ch >= d.in_off && ch < d.in_off + d.c_in) v = 0.0f;
                gg[it][c] = v;
                // bf16 cells: dx is a bf16 tensor, so its gradient is bf16
                gd[c] = ok ? rnd<BF16>(v * f) : 0.0f;
            }
            if (BF16) {
                put4<BF16>(GDL + (n * S::DS + c0) * S::ES, gd);
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) reinterpret_cast<float *>(GDL)[n * S::DS + S::col(c0 + c)] = gd[c];
            }
        }
        if (has_loss) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int p = tid + 256 * s;
                if (p < np) {
                    const int v = p < npw ? p / d.c_out : p - npw, c = p < npw ? p - v * d.c_out : -1;
#pragma unroll 8
                    for (int n = 0; n < kBN; ++n) hs[s] = __builtin_fmaf(glL[n][v], c < 0 ? 1.0f : xoL[n][c < 0 ? 0 : c], hs[s]);
                }
            }
            if (tid == 255)
#pragma unroll
                for (int n = 0; n < kBN; ++n) lossv = __fadd_rn(lossv, lossL[n]);
        }
        __syncthreads();
        // ---- h and g_a: wave w, hidden units [w HD / 4, (w + 1) HD / 4)
        WFrags<BF16, S::MT2, S::KH> w1t;
        {
            nca::f32x4 h[S::MT1][2], ga[S::MT1][2];
#pragma unroll
            for (int m = 0; m < S::MT1; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n) h[m][n] = ga[m][n] = nca::f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            w1.mma(ZL, S::ZS * S::ES, lane, h);
            w2t.mma(GDL, S::DS * S::ES, lane, ga);
            w1t.load(a.w1t, wave * S::MT2, lane);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < S::MT1; ++m) {
                const int hid = (wave * S::MT1 + m) * 16 + 4 * g;
                const float4 b4 = *reinterpret_cast<const float4 *>(a.b1 + hid);
                const float bb[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const int cell = 16 * n + l16;
                    float hr[4], gv[4];
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float hv = rnd<BF16>(__fadd_rn(h[m][n][v], bb[v]));
                        hr[v] = hv > 0.0f ? hv : 0.0f;
                        gv[v] = hr[v] > 0.0f ? rnd<BF16>(ga[m][n][v]) : 0.0f;
                    }
                    if (BF16) {
                        put4<BF16>(HL + (cell * S::GS + hid) * S::ES, hr);
                        put4<BF16>(GAL + (cell * S::GS + hid) * S::ES, gv);
                    } else {
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            reinterpret_cast<float *>(GAL)[cell * S::GS + S::col(hid + v)] = gv[v];
                            static_cast<float *>(a.hs)[((a.tile0 + tile) * HD + hid + v) * kBN + cell] = hr[v];
                        }
                    }
                }
            }
        }
        __syncthreads();
        // ---- g_z: wave w, features [w F / 4, (w + 1) F / 4)
        {
            nca::f32x4 gz[S::MT2][2];
#pragma unroll
            for (int m = 0; m < S::MT2; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n) gz[m][n] = nca::f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            w1t.mma(GAL, S::GS * S::ES, lane, gz);
#pragma unroll
            for (int m = 0; m < S::MT2; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const float v[4] = {gz[m][n][0], gz[m][n][1], gz[m][n][2], gz[m][n][3]};
                    put4<BF16>(GZL + ((16 * n + l16) * S::ZS + (wave * S::MT2 + m) * 16 + 4 * g) * S::ES, v);
                }
        }
        __syncthreads();
        // ---- the kernel-weight sums (the taps again, from the caches), folded over rows of 16 lanes
        {
            float dk[36];
#pragma unroll
            for (int v = 0; v < 36; ++v) dk[v] = 0.0f;
#pragma unroll
            for (int it = 0; it < S::NZ; ++it) {
                const int e = tid + 256 * it, n = e & (kBN - 1), c0 = 4 * (e / kBN);
                if (e >= S::ITEMS || m0 + n >= M) continue;
                float xv[4][9];
                cell_taps<C, BF16>(d, a.xt, a.padv, rowL[n], iL[n], jL[n], c0, xv);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float gv[4];
                    get4<BF16>(GZL + (n * S::ZS + k * C + c0) * S::ES, gv);
#pragma unroll
                    for (int c = 0; c < 4; ++c)
#pragma unroll
                        for (int t = 0; t < 9; ++t) dk[k * 9 + t] = __builtin_fmaf(gv[c], xv[c][t], dk[k * 9 + t]);
                }
            }
#pragma unroll
            for (int v = 0; v < 36; ++v) {
                float x = dk[v];
                x = __fadd_rn(x, dpp_f32<0xb1>(x));
                x = __fadd_rn(x, dpp_f32<0x4e>(x));
                x = __fadd_rn(x, dpp_f32<0x141>(x));
                x = __fadd_rn(x, dpp_f32<0x140>(x));
                if (l16 == 0) red[(tid >> 4) * 36 + v] = __fadd_rn(red[(tid >> 4) * 36 + v], x);
            }
        }
        // ---- everything out: stores last, so that no load of the tile waits behind them (they
        // complete in order with the loads)
#pragma unroll
        for (int it = 0; it < S::NZ; ++it) {
            const int e = tid + 256 * it, c0 = 4 * (e & (C / 4 - 1)), n = e / (C / 4);
            if (e < S::ITEMS && m0 + n < M)
                *reinterpret_cast<float4 *>(a.f.Gu + (int64_t)(m0 + n) * C + c0) =
                    make_float4(gg[it][0], gg[it][1], gg[it][2], gg[it][3]);
        }
        constexpr int UPR = S::F * S::ES / 16;  // 16-byte units per cell of g_z
        for (int u = tid; u < kBN * UPR; u += 256) {
            const int n = u / UPR, o = u - n * UPR;
            if (m0 + n < M)
                reinterpret_cast<uint4 *>(a.gz_out)[(int64_t)(m0 + n) * UPR + o] =
                    *reinterpret_cast<const uint4 *>(GZL + n * S::ZS * S::ES + 16 * o);
        }
        flush_tile<S, BF16, true>(ZL, S::ZS, S::F, a.zs, a.tile0 + tile);
        if (BF16) flush_tile<S, BF16, false>(HL, S::GS, HD, a.hs, a.tile0 + tile);
        flush_tile<S, BF16, true>(GAL, S::GS, HD, a.gas, a.tile0 + tile);
        flush_tile<S, BF16, true>(GDL, S::DS, C, a.gds, a.tile0 + tile);
        __syncthreads();
    }
    // ---- the workgroup's slots
    float *sl = a.slots + (int64_t)blockIdx.x * a.nslot;
    if (tid < 36) {
        float r = a.accum ? sl[tid] : 0.0f;
#pragma unroll
        for (int w = 0; w < 16; ++w) r = __fadd_rn(r, red[w * 36 + tid]);  // the 16 lane rows in order
        sl[tid] = r;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int p = tid + 256 * s;
        if (p < np) sl[36 + p] = a.accum ? __fadd_rn(sl[36 + p], hs[s]) : hs[s];
    }
    if (tid == 255) sl[36 + np] = a.accum ? __fadd_rn(sl[36 + np], lossv) : lossv;
}

// The gradient of the chunk's first state, (rows, C, H, W), from the first step's g_u and g_z.
template <int C, bool BF16>
__global__ void __launch_bounds__(256) back_x0(Dims d, const float *Gu, const void *Gz, const float *kern, float *gx) {
    const int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x;  // (cell, channel quad), quads fastest
    const int64_t m = e / (C / 4);
    if (m >= d.M) return;
    const int c0 = 4 * (int)(e - m * (C / 4));
    const int64_t row = m / d.HW;
    const int q = (int)(m - row * d.HW), i = q / d.W, j = q - i * d.W;
    float g[4];
    later_grad<C, BF16>(d, Gu, Gz, kern, row * d.HW, i, j, c0, g);
#pragma unroll
    for (int c = 0; c < 4; ++c) gx[(row * C + c0 + c) * (int64_t)d.HW + q] = g[c];
}

struct WeightGradArgs {
    const unsigned char *ga, *z, *gd, *h;  // [tile][feature][32 cells]
    int64_t K, kps;  // tiles in use, per split
    int C, F, HD, splits;
    float *part;         // slot s: part + s P
    int64_t P, offW1, offB1, offW2, offB2;
    int accum;
};

// dW1 (HD x F) = g_a z^T, dW2 (C x HD) = g_dx h^T and the row sums db1 of g_a and db2 of g_dx over
// the tiles [s kps, (s + 1) kps): a workgroup takes a 128 x 64 tile of dW1 (or up to 64 x 64 of
// dW2), wave w its 64 x 32 part, for one s. A lane's 16 bytes of a tile's row are its MFMA
// operand as they lie: no LDS. The kernel reads its operands once per
// tile of the other one, so it is bound by those reads; the workgroups of one s have the same index
// modulo 8, hence the same XCD and L2.
template <bool BF16>
__global__ void __launch_bounds__(256, 3) weight_grads(WeightGradArgs a) {
    typedef typename BFrag<BF16>::type fr;
    constexpr int ES = BF16 ? 2 : 4, KT = kBN * ES / 64;  // k-blocks (64 bytes of a row) per tile
    constexpr int RA = 4, RB = 2;                   // 16-row blocks of A and B per wave
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, l16 = lane & 15;
    const int nt1 = a.F / 64, t1 = (a.HD / 128) * nt1, nt = t1 + a.HD / 64;
    const int grp = blockIdx.x / (8 * nt), rem = blockIdx.x - grp * 8 * nt;
    const int t = rem >> 3, split = grp * 8 + (rem & 7);
    if (split >= a.splits) return;
    const bool first = t < t1;
    const int tt = first ? t : t - t1;
    const int ti = first ? tt / nt1 : 0, tj = first ? tt - ti * nt1 : tt;
    const int r0 = 128 * ti + 64 * (wave >> 1), c0 = 64 * tj + 32 * (wave & 1);
    const int rows = first ? a.HD : a.C, ldo = first ? a.F : a.HD;
    const unsigned char *A = first ? a.ga : a.gd, *B = first ? a.z : a.h;
    if (r0 >= rows) return;  // dW2 has at most 64 rows
    const int nr = rows - r0 < 64 ? (rows - r0) / 16 : RA;  // row blocks in use
    const bool bias = tj == 0 && (wave & 1) == 0;
    // in k-blocks
    const int64_t k0 = split * a.kps * KT, k1 = (split + 1) * a.kps < a.K ? k0 + a.kps * KT : a.K * KT;
    const int64_t ta = (int64_t)rows * kBN * ES, tb = (int64_t)ldo * kBN * ES;  // bytes per tile
    const unsigned char *pa[RA], *pb[RB];
#pragma unroll
    for (int r = 0; r < RA; ++r) pa[r] = A + (r0 + 16 * (r < nr ? r : 0) + l16) * kBN * ES + 16 * g;
#pragma unroll
    for (int r = 0; r < RB; ++r) pb[r] = B + (c0 + 16 * r + l16) * kBN * ES + 16 * g;
    nca::f32x4 acc[RA][RB], ab[RA];
#pragma unroll
    for (int r = 0; r < RA; ++r) {
        ab[r] = nca::f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < RB; ++c) acc[r][c] = nca::f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    fr ones;
#pragma unroll
    for (int i = 0; i < 16 / ES; ++i) ones[i] = 1.0f;
    constexpr int U = 2;  // k-blocks in flight
    uint4 va[U][RA], vb[U][RB];
    auto load = [&](int u, int64_t k) {
        const int64_t kk = k < k1 ? k : k0;  // a block past the range: loaded, not used
        const int64_t oa = kk / KT * ta + kk % KT * 64, ob = kk / KT * tb + kk % KT * 64;
#pragma unroll
        for (int r = 0; r < RA; ++r) va[u][r] = *reinterpret_cast<const uint4 *>(pa[r] + oa);
#pragma unroll
        for (int r = 0; r < RB; ++r) vb[u][r] = *reinterpret_cast<const uint4 *>(pb[r] + ob);
    };
    if (k0 < k1) {
        load(0, k0);
        load(1, k0 + 1);
    }
    for (int64_t k = k0; k < k1; k += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k + u < k1) {  // uniform
#pragma unroll
                for (int r = 0; r < RA; ++r) {
                    const fr av = __builtin_bit_cast(fr, va[u][r]);
#pragma unroll
                    for (int c = 0; c < RB; ++c) acc[r][c] = BFrag<BF16>::mma(av, __builtin_bit_cast(fr, vb[u][c]), acc[r][c]);
                    if (bias) ab[r] = BFrag<BF16>::mma(av, ones, ab[r]);
                }
            }
            load(u, k + U + u);
        }
    }
    float *out = a.part + (int64_t)split * a.P + (first ? a.offW1 : a.offW2);
    float *ob = a.part + (int64_t)split * a.P + (first ? a.offB1 : a.offB2);
#pragma unroll
    for (int r = 0; r < RA; ++r) {
        if (r >= nr) break;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int row = r0 + 16 * r + 4 * g + v;
#pragma unroll
            for (int c = 0; c < RB; ++c) {
                float *p = out + (int64_t)row * ldo + c0 + 16 * c + l16;
                *p = a.accum ? __fadd_rn(*p, acc[r][c][v]) : acc[r][c][v];
            }
            if (bias && l16 == 0) ob[row] = a.accum ? __fadd_rn(ob[row], ab[r][v]) : ab[r][v];
        }
    }
}

// The chunk's gradients out of the slots: thread per MLP parameter (`splits` slots of part, in slot
// order), wave per kernel weight, head parameter and the loss (`wgs` slots, lanes strided, then a
// fixed fold). `nbig` workgroups do the former.
__global__ void __launch_bounds__(256) back_finish(const float *part, int64_t P, int splits, const float *slots, int nslot,
                                                   int wgs, int nbig, int64_t offK, int64_t lo, int64_t hi, int64_t offHW,
                                                   GradOut go, float *loss_out) {
    if ((int)blockIdx.x < nbig) {
        const int64_t i = lo + blockIdx.x * (int64_t)256 + threadIdx.x;
        if (i >= hi) return;
        constexpr int kB = 32;
        float s = 0.0f;
        for (int k0 = 0; k0 < splits; k0 += kB) {
            float v[kB];
#pragma unroll
            for (int k = 0; k < kB; ++k) v[k] = k0 + k < splits ? part[(int64_t)(k0 + k) * P + i] : 0.0f;
#pragma unroll
            for (int k = 0; k < kB; ++k)
                if (k0 + k < splits) s = __fadd_rn(s, v[k]);
        }
#pragma unroll
        for (int k = 0; k < 7; ++k)
            if (go.dst[k] && i >= go.off[k] && i < go.off[k] + go.n[k]) grad_put(go, k, i - go.off[k], s);
        return;
    }
    const int v = (blockIdx.x - nbig) * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (v >= nslot) return;
    float s = 0.0f;
    for (int w = lane; w < wgs; w += 64) s = __fadd_rn(s, slots[(int64_t)w * nslot + v]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s = __fadd_rn(s, __shfl_xor(s, o));
    if (lane != 0) return;
    if (v == nslot - 1) {
        if (loss_out) *loss_out = s;
        return;
    }
    const int64_t i = v < 36 ? offK + v : offHW + (v - 36);
#pragma unroll
    for (int k = 0; k < 7; ++k)
        if (go.dst[k] && i >= go.off[k] && i < go.off[k] + go.n[k]) grad_put(go, k, i - go.off[k], s);
}

}  // namespace
