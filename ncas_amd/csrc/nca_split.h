// fp32 products on the bf16 matrix cores (gfx950): every fp32 operand is held as three bf16
// values, v = h + m + l with h = bf16(v), m = bf16(v - h), l = bf16(v - h - m) (round to nearest
// even; 3 x 8 significand bits hold all 24), and a product takes the six largest of the nine
// partial products (l l, l m and m l lie below 2^-24 of it, the rounding of one fp32 product).
// bf16 products are exact in fp32 and MFMA accumulates in fp32, so a dot product's error is that
// of an fp32 chain or less: a step's relative error against 64 bits is 4.1e-8 to 5.2e-8 (C = 16,
// boards of 13x13 to 40x40), 6.7e-8 to 8.5e-8 with fp32 MFMA.
// v_mfma_f32_16x16x32_bf16 does 32 k in 16 cycles, v_mfma_f32_16x16x4_f32 4 k in 32: six of
// the former cost 96 cycles where eight of the latter cost 256. (VALU work adds to that more than
// it does beside other MFMAs: an MFMA of this form holds the SIMD's issue port for about 11 of
// its 16 cycles, measured with one MFMA and one VALU wave per SIMD. v_mfma_f32_32x32x16_bf16 does
// not, but its 32-cell tiles leave 8 waves per CU, and their waits cost what it saves: 201x201
// steps 98 us in both forms, 13x13 rollouts 2.40 ms against 1.87.)
//
// The exponent range is fp32's, but parts below bf16's least value, 2^-133, are lost: values below 2^-109
// keep fewer than 24 bits. A value that rounds to an infinite h (or is infinite or NaN) makes
// m or l NaN, hence every output of its cell: a tile with a NaN among fc1's or fc2's sums is
// computed again on fp32 MFMA (a branch uniform over the wave), and the cells with a NaN of their
// own take that result, so infinities and NaN come out as they do there. An MFMA's columns
// are its cells and do not mix: the tile's other cells keep theirs, so that a cell's
// bits do not depend on which cells share its tile.
#pragma once

#include "nca_rollout.h"
#include "nca_stream_util.h"

namespace nca {

// v - the low / high half of a bf16 pair, one v_dot2_f32_bf16 (an unpacking shift and a subtraction
// otherwise). With h = bf16(v) the difference is an fp32 value, so the sum's rounding does not
// matter; an infinite or NaN half makes both differences NaN. The pairs (-1, 0) and (0, -1) come
// from registers: as the instruction's inline constant -1.0 the former is read as the latter.
__device__ __forceinline__ uint32_t bf16_const(uint32_t v) {
    asm("" : "+s"(v));
    return v;
}
__device__ __forceinline__ float minus_lo(float v, uint32_t h) {
    return __builtin_amdgcn_fdot2_f32_bf16(as_bf16x2(h), as_bf16x2(bf16_const(0x0000bf80u)), v, false);
}
__device__ __forceinline__ float minus_hi(float v, uint32_t h) {
    return __builtin_amdgcn_fdot2_f32_bf16(as_bf16x2(h), as_bf16x2(bf16_const(0xbf800000u)), v, false);
}
// two floats -> the packed bf16 pairs of their three parts
__device__ __forceinline__ void split3(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l) {
    h = cvt_pk_bf16(a, b);
    const float ra = minus_lo(a, h), rb = minus_hi(b, h);
    m = cvt_pk_bf16(ra, rb);
    l = cvt_pk_bf16(minus_lo(ra, m), minus_hi(rb, m));
}

// max(v, 0) in one instruction (v is no NaN where the result is used)
__device__ __forceinline__ float relu_f32(float v) { return __builtin_amdgcn_fmed3f(v, 0.0f, INFINITY); }

// a B operand (8 k slots of the lane's cell) in three parts
struct Split8 {
    uint4 h, m, l;
};
__device__ __forceinline__ Split8 split8(const float v[8]) {
    Split8 s;
    split3(v[0], v[1], s.h.x, s.m.x, s.l.x);
    split3(v[2], v[3], s.h.y, s.m.y, s.l.y);
    split3(v[4], v[5], s.h.z, s.m.z, s.l.z);
    split3(v[6], v[7], s.h.w, s.m.w, s.l.w);
    return s;
}

__device__ __forceinline__ f32x4 mfma_bf(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// the three smallest, the two middle and the largest partial products of a k-block
__device__ __forceinline__ f32x4 mfma_small(const Split8 &w, const Split8 &v, f32x4 c) {
    c = mfma_bf(w.l, v.h, c);
    c = mfma_bf(w.h, v.l, c);
    return mfma_bf(w.m, v.m, c);
}
__device__ __forceinline__ f32x4 mfma_mid(const Split8 &w, const Split8 &v, f32x4 c) {
    c = mfma_bf(w.m, v.h, c);
    return mfma_bf(w.h, v.m, c);
}

// ------------------------------------------------------------------------------------------
// The C = 16, 128-hidden cell's MLP of one 16-cell tile, by one wave: lane (cell r = lane & 15, g =
// lane >> 4) brings z of its cell's channels 4 g .. 4 g + 3 for the 4 kernels and gets dx of the
// same channels. Both products' k orders are permuted (in the packed weights) so that z, and
// fc1's accumulators, are the B operands as they lie in the lane: nothing passes through LDS
// but the weights (60 KB for the workgroup), 16 bytes a lane per fragment.
constexpr int kSplit16Frags = 8 * 2 * 3 + 4 * 3;  // [m-tile][k-tile][part] of W1, [k-tile][part] of W2
constexpr unsigned kSplit16Bytes = kSplit16Frags * 1024u;

__device__ __forceinline__ Split8 lds_frag3(const unsigned char *wl, int first, int lane) {
    const uint4 *p = reinterpret_cast<const uint4 *>(wl) + first * 64 + lane;
    return Split8{p[0], p[64], p[128]};
}

// fp32 MFMA on the forward's packed fp32 fragments (global memory): tiles that hold a NaN
__device__ __forceinline__ f32x4 mlp16_fp32(const float z[4][4], const float *w1, const float *w2, const float *b1L, f32x4 b2v,
                                            int lane) {
    const int g = lane >> 4, l16 = lane & 15;
    f32x4 dx = b2v;
#pragma unroll 1
    for (int mt = 0; mt < 8; ++mt) {
        const float4 bq = *reinterpret_cast<const float4 *>(b1L + 16 * mt + 4 * g);
        f32x4 h = {bq.x, bq.y, bq.z, bq.w};
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                h = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[((mt * 4 + k) * 64 + 16 * c + l16) * 4 + g], z[k][c], h, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; ++v)
            dx = __builtin_amdgcn_mfma_f32_16x16x4f32(w2[(4 * mt + g) * 64 + 16 * v + l16], h[v] > 0.0f ? h[v] : 0.0f, dx, 0, 0, 0);
    }
    return dx;
}

__device__ __forceinline__ f32x4 mlp16_split(const float z[4][4], const unsigned char *wl, const float *b1L, f32x4 b2v,
                                             const float *w1, const float *w2, int lane) {
    const int g = lane >> 4;
    Split8 zs[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
        const float v[8] = {z[2 * kt][0],     z[2 * kt][1],     z[2 * kt][2],     z[2 * kt][3],
                            z[2 * kt + 1][0], z[2 * kt + 1][1], z[2 * kt + 1][2], z[2 * kt + 1][3]};
        zs[kt] = split8(v);
    }
    // the largest products of even and odd k-tiles and the smaller ones in sums of their own: a rounding
    // of a smaller sum costs less
    bool bad = false;
    f32x4 dl[2] = {b2v, f32x4{0.0f, 0.0f, 0.0f, 0.0f}}, ds = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        f32x4 h[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int mt = 2 * j + i;
            const float4 bq = *reinterpret_cast<const float4 *>(b1L + 16 * mt + 4 * g);
            const Split8 w0 = lds_frag3(wl, (2 * mt) * 3, lane), w1s = lds_frag3(wl, (2 * mt + 1) * 3, lane);
            f32x4 c = {bq.x, bq.y, bq.z, bq.w};
            c = mfma_small(w0, zs[0], c);
            c = mfma_small(w1s, zs[1], c);
            c = mfma_mid(w0, zs[0], c);
            c = mfma_mid(w1s, zs[1], c);
            c = mfma_bf(w0.h, zs[0].h, c);
            h[i] = mfma_bf(w1s.h, zs[1].h, c);
        }
        float hv[8];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            bad |= __builtin_isunordered(h[i][0], h[i][1]) | __builtin_isunordered(h[i][2], h[i][3]);
#pragma unroll
            for (int v = 0; v < 4; ++v) hv[4 * i + v] = relu_f32(h[i][v]);
        }
        const Split8 hs = split8(hv), w2s = lds_frag3(wl, 48 + 3 * j, lane);
        ds = mfma_small(w2s, hs, ds);
        ds = mfma_mid(w2s, hs, ds);
        dl[j & 1] = mfma_bf(w2s.h, hs.h, dl[j & 1]);
    }
    f32x4 dx = (dl[0] + dl[1]) + ds;
    bad |= __builtin_isunordered(dx[0], dx[1]) | __builtin_isunordered(dx[2], dx[3]);
    const uint64_t nan = __ballot(bad);
    if (nan) {
        const uint64_t cells = nan | nan >> 16 | nan >> 32 | nan >> 48;  // bits 0..15: over the cell's four lanes
        const f32x4 d = mlp16_fp32(z, w1, w2, b1L, b2v, lane);
        const bool own = (cells >> (lane & 15)) & 1;
#pragma unroll
        for (int v = 0; v < 4; ++v) dx[v] = own ? d[v] : dx[v];
    }
    return dx;
}

// z of the lane's 4 channels from their 9 taps (the tap chains of the other fp32 kernels)
__device__ __forceinline__ void stencil16(const f32x4 tp[9], const float *kern, float z[4][4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int c = 0; c < 4; ++c) z[k][c] = 0.0f;
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float w = kern[k * 9 + t];
#pragma unroll
            for (int c = 0; c < 4; ++c) z[k][c] = __builtin_fmaf(w, tp[t][c], z[k][c]);
        }
}

struct Split16Step {
    RolloutParams a;  // x_in -> x_out of this step (distinct buffers); fire_u8: this step's masks
    const unsigned char *wsplit;
    int step;         // step index within the call (Philox counter step0 + step)
    int64_t n_tiles;  // rows * tiles_per_row
    int tiles_per_row;
    int64_t tiles_per_wg;
};

struct Split16Resident {
    RolloutParams a;
    const unsigned char *wsplit;
    int R;  // rows per workgroup
    unsigned l_P, l_ci, l_fire, l_given, l_fired, l_head, total;
};

}  // namespace nca
