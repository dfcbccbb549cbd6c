// One head row of the per-token Q/K/V preparation: bias, QK RMSNorm, RoPE, Gemma q scale, in
// f32.  The body of the preparation kernel (qkv_prep.hip) and of the Turbo cache's fused
// token kernel (turbo_decode.hip), which must round a row alike.
#pragma once

#include "gr_common.hpp"
#include "gr_internal.hpp"

namespace gr {

// 8 consecutive elements (one 16-byte chunk of a 16-bit row, two of an f32 row).
__device__ __forceinline__ void load8(const void* base, size_t idx, int dt, float* v) {
    if (dt == GR_DTYPE_F32) {
        const float4 a = *(const float4*)((const float*)base + idx);
        const float4 b = *(const float4*)((const float*)base + idx + 4);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
        return;
    }
    const uint4 u = *(const uint4*)((const uint16_t*)base + idx);
    if (dt == GR_DTYPE_F16) unpack16<F16>(u, v);
    else unpack16<BF16>(u, v);
}

// The token's RoPE cos / sin (the rebuild_rope_cache angle (pos*freq)*scale): frequencies
// f0, f0 + step, .. into cs_t / sn_t and, when cs_out is set, as pairs to cs_out.
__device__ __forceinline__ void prep_rope_table(const QkvPrepLaunch& p, int64_t pos, int f0, int step, float* cs_t,
                                                float* sn_t, float* cs_out) {
    for (int f = f0; f < p.rope_dim / 2; f += step) {
        const float val = ((float)pos * p.rope_freqs[f]) * p.rope_scale;
        float sn, cs;
        sincosf(val, &sn, &cs);
        cs_t[f] = cs;
        sn_t[f] = sn;
        if (cs_out) *(float2*)(cs_out + 2 * f) = make_float2(cs, sn);
    }
}

// Elements c8 .. c8 + 7 of row `head` of kind 0 (q), 1 (k) or 2 (v) of token i: D / 8
// consecutive lanes hold a row, `rb` is [D] floats of LDS of that lane group; every lane of
// the wave runs it (the row sums).  The sums of products are spelled out as fused
// operations: left to contraction, two kernels may round them differently, and a row one
// rounding off can take other codes in a quantised cache.  Launch and row by value: by
// reference the prep kernel takes 84 registers instead of 79, five waves per SIMD instead
// of six (8192 tokens, 32 / 8 heads of 128: 28 us with five, 21 with six).
struct PrepRow {
    float x[8];
};
template <int D>
__device__ __forceinline__ PrepRow prep_row(const QkvPrepLaunch p, int i, int kind, int head, int c8,
                                            const float* cs_t, const float* sn_t, float* rb) {
    PrepRow row;
    float (&x)[8] = row.x;
    constexpr int LPR = D / 8;  // lanes per row
    const bool rope = p.rope_mode != GR_ROPE_NONE;
    const int half = p.rope_dim / 2;
    const void* src = kind == 0 ? p.q : (kind == 1 ? p.k : p.v);
    const int64_t rs = kind == 0 ? p.q_row_stride : p.kv_row_stride;
    load8(src, (size_t)i * rs + (size_t)head * D + c8, p.in_dtype, x);
    // Qwen2 attention biases, before the norm (qkv_bias_and_norm, inference.rs:2545-2559)
    const float* bias = kind == 0 ? p.q_bias : (kind == 1 ? p.k_bias : p.v_bias);
    if (bias) {
        float bv[8];
        load8(bias, (size_t)head * D + c8, GR_DTYPE_F32, bv);
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] += bv[e];
    }
    if (kind != 2) {
        // QK RMSNorm: ss = sum(x^2)/d + eps; x = w * ((1/sqrt(ss)) * x).
        const float* w = kind == 0 ? p.q_norm : p.k_norm;
        float ss = fmaf(x[0], x[0], x[1] * x[1]);
#pragma unroll
        for (int e = 2; e < 8; e++) ss = fmaf(x[e], x[e], ss);
        ss = wave_sum<LPR>(ss);  // lanes of other rows never mix: groups are LPR-aligned
        if (w) {
            const float inv = 1.0f / sqrtf(ss / (float)D + p.eps);
            float wv[8];
            load8(w, c8, GR_DTYPE_F32, wv);
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = wv[e] * (inv * x[e]);
        }
        if (rope) {
            if (p.rope_mode == GR_ROPE_ADJACENT) {
                // pairs (2j, 2j+1) sit inside the lane's 8 elements
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const int fi = (c8 + e) >> 1;
                    const float cs = cs_t[fi], sn = sn_t[fi];
                    const float v0 = x[e], v1 = x[e + 1];
                    x[e] = fmaf(v0, cs, -(v1 * sn));
                    x[e + 1] = fmaf(v1, cs, v0 * sn);
                }
            } else if (p.rope_dim == D) {
                // NeoX pairs (i, i + D/2) of a fully rotated row: the partner
                // elements of this lane's 8 are the 8 of lane ^ (LPR/2), in the
                // same row's lane group
                const bool first = c8 < half;
                const int f0 = first ? c8 : c8 - half;
                float csv[8], snv[8];
                *(float4*)csv = *(const float4*)(cs_t + f0);
                *(float4*)(csv + 4) = *(const float4*)(cs_t + f0 + 4);
                *(float4*)snv = *(const float4*)(sn_t + f0);
                *(float4*)(snv + 4) = *(const float4*)(sn_t + f0 + 4);
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float other = __shfl_xor(x[e], LPR / 2, 64);
                    // (v0, v1) -> (v0*c - v1*s, v0*s + v1*c)
                    x[e] = first ? fmaf(-other, snv[e], x[e] * csv[e]) : fmaf(other, snv[e], x[e] * csv[e]);
                }
            } else {
                // NeoX pairs (i, i + rope_dim/2) of a partial rotation live in
                // other lanes: stage the row
#pragma unroll
                for (int e = 0; e < 8; e++) rb[c8 + e] = x[e];
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int idx = c8 + e;
                    if (idx >= p.rope_dim) continue;  // partial RoPE: tail untouched
                    const bool first = idx < half;
                    const int fi = first ? idx : idx - half;
                    const float other = rb[first ? idx + half : idx - half];
                    const float cs = cs_t[fi], sn = sn_t[fi];
                    // (v0, v1) -> (v0*c - v1*s, v0*s + v1*c)
                    x[e] = first ? fmaf(x[e], cs, -(other * sn)) : fmaf(x[e], cs, other * sn);
                }
                __builtin_amdgcn_wave_barrier();  // reads done before the next rows' stores
            }
        }
        if (kind == 0 && p.gemma_q_scale) {
            const float sc = 1.0f / sqrtf((float)D);
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] *= sc;
        }
    }
    return row;
}

}  // namespace gr
