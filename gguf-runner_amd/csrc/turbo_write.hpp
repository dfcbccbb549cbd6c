// The quantising write of one (row, kv head, K|V) of a Turbo cache by one wave
// (quantize_turboquant_head, inference.rs:855-925), shared by the write kernel
// (turbo.hip) and the fused token kernel (turbo_decode.hip).  No FMA contraction: the
// codes, signs, sigma and gamma are bit-exact with the reference for the same row.
#pragma once

#include "gr_common.hpp"
#include "gr_internal.hpp"
#include "turbo_common.hpp"

namespace gr {

__device__ __forceinline__ float tq_centroid(int code) {
    return code == 0 ? -tq::kC1 : code == 1 ? -tq::kC0 : code == 2 ? tq::kC0 : tq::kC1;
}

__device__ __forceinline__ int tq_code(float x) {
    return x < -tq::kTh ? 0 : (x < 0.0f ? 1 : (x < tq::kTh ? 2 : 3));
}

// l2_norm (math.rs:467-473): sequential sum in element order, every lane the same
template <int D>
__device__ __forceinline__ float wave_l2_sequential(const float (&x)[D / 64], float* buf, int lane) {
#pragma clang fp contract(off)
#pragma unroll
    for (int j = 0; j < D / 64; j++) buf[lane + 64 * j] = x[j];
    tq::wave_lds_sync();
    float ss = 0.0f;
    for (int e = 0; e < D; e++) {
        const float v = buf[e];
        ss = ss + v * v;
    }
    tq::wave_lds_sync();  // buf is reused by the caller
    return sqrtf(ss);
}

// x: the row, element lane + 64 j; destination row i of the launch; buf [D] floats and
// codes [D] bytes of LDS of this wave.
template <int D>
__device__ __forceinline__ void turbo_write_unit(const TurboWriteLaunch& p, int i, int g, bool is_v,
                                                 float (&x)[D / 64], float* buf, uint8_t* codes, int lane) {
#pragma clang fp contract(off)
    constexpr int J = D / 64;
    const int64_t row = p.cache_row ? (int64_t)p.cache_row[i] : p.row0 + i;
    const int64_t sq = p.cache_seq ? (int64_t)p.cache_seq[i] : 0;
    const int64_t elem = sq * p.cache_seq_stride + row * p.cache_row_stride + (int64_t)g * D;
    uint8_t* base = (is_v ? p.v_base : p.k_base) + elem / 4;
    uint8_t* sign = (is_v ? p.v_sign : p.k_sign) + elem / 8;
    const int64_t aux = sq * p.aux_seq_stride + row * p.aux_row_stride + g;
    float* scale_out = (is_v ? p.v_scale : p.k_scale) + aux;
    float* rnorm_out = (is_v ? p.v_rnorm : p.k_rnorm) + aux;
    const uint8_t* sg = p.signs + (size_t)g * (D / 8);
    const int64_t ss = p.slot_stride;
    tq::wave_transform<D>(x, sg, sg + ss, lane);  // rot_pre, rot_post
    const float sigma = wave_l2_sequential<D>(x, buf, lane) / sqrtf((float)D);
    if (sigma == 0.0f) {
        if (lane == 0) {
            *scale_out = 0.0f;
            *rnorm_out = 0.0f;
        }
        if (lane < D / 4) base[lane] = 0;
        if (lane < D / 8) sign[lane] = 0xff;
        return;
    }
    const float inv_sigma = 1.0f / sigma;
    float r[J];
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int c = tq_code(x[j] * inv_sigma);
        r[j] = x[j] - tq_centroid(c) * sigma;
        codes[lane + 64 * j] = (uint8_t)c;
    }
    const float gamma = wave_l2_sequential<D>(r, buf, lane);  // its first synchronisation also publishes `codes`
    if (lane < D / 4)
        base[lane] = (uint8_t)(codes[4 * lane] | (codes[4 * lane + 1] << 2) | (codes[4 * lane + 2] << 4) |
                               (codes[4 * lane + 3] << 6));
    if (lane == 0) {
        *scale_out = sigma;
        *rnorm_out = gamma;
    }
    if (gamma == 0.0f) {
        if (lane < D / 8) sign[lane] = 0xff;
        return;
    }
#pragma unroll
    for (int j = 0; j < J; j++) r[j] = r[j] / gamma;
    tq::wave_transform<D>(r, sg + 2 * ss, sg + 3 * ss, lane);  // res_pre, res_post
#pragma unroll
    for (int j = 0; j < J; j++) {
        const uint64_t m = __ballot(r[j] >= 0.0f);  // bit l = element 64 j + l
        if (lane == 0) *(uint64_t*)(sign + 8 * j) = m;
    }
}

}  // namespace gr
