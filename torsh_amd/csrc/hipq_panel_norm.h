// LayerNorm + per-token int8 of a row by one wave with the bits of the row-panel GEMM's epilogue (hipq_gemm_rows.h): its sums
// run over a lane's column blocks first, then over the 32 columns of a block (neighbours first), then over the eight waves in
// pairs, and in the pair form over the two halves of the columns last.  Eight lanes stand for a panel wave here, four
// neighbouring columns each, so the panel's fold is this wave's butterfly in ascending order and a load is 16 bytes a lane.
// RC float4 a lane; PAIR: the first RC / 2 of them belong to the first half of the columns.
#pragma once

#include "hipq_internal.h"
#include "hipq_math.h"

namespace hipq {

template <int RC, bool PAIR>
struct PanelColumns {  // the lane's columns: part * 4 .. + 3 of the blocks of 32 that are real
    int block[RC], part, cols;
    bool real[RC];
    __device__ __forceinline__ PanelColumns(int lane, int nblocks) : part(lane % 8), cols(nblocks * 32) {
        constexpr int H = PAIR ? 2 : 1, PER = RC / H;
        const int wave = lane / 8, half_blocks = nblocks / H;
#pragma unroll
        for (int i = 0; i < RC; ++i) {
            const int b = PAIR ? wave + 8 * (i % PER) : wave * RC + i;
            real[i] = b < half_blocks;
            block[i] = b + (i / PER) * half_blocks;
        }
    }
    __device__ __forceinline__ int at(int i) const { return block[i] * 32 + part * 4; }
};

// Gain and offset of a lane's columns.
template <int RC>
struct PanelAffine {
    float4 g[RC], b[RC];
    __device__ __forceinline__ PanelAffine() {}
    template <bool PAIR>
    __device__ __forceinline__ PanelAffine(const PanelColumns<RC, PAIR> &c, const float *gamma, const float *beta) {
        auto affine = [&](const float *p, int i, float missing) {
            if (!p || !c.real[i]) return make_float4(missing, missing, missing, missing);
            const AnyFloat4 t = *reinterpret_cast<const AnyFloat4 *>(p + c.at(i));
            return make_float4(t.x, t.y, t.z, t.w);
        };
#pragma unroll
        for (int i = 0; i < RC; ++i) {  // (y * 1.0f and y + -0.0f are y, bit for bit)
            g[i] = affine(gamma, i, 1.0f);
            b[i] = affine(beta, i, -0.0f);
        }
    }
};

// v: the row, replaced by its normalized values; q[i]: the codes of v[i] (of real blocks).  Returns the row's scale.
template <bool EVEN, int RC, bool PAIR>
__device__ __forceinline__ float panel_norm_quantize(float4 (&v)[RC], const PanelColumns<RC, PAIR> &c, const PanelAffine<RC> &a,
                                                     float eps, uint32_t (&q)[RC]) {
    constexpr int H = PAIR ? 2 : 1, PER = RC / H;
    auto total = [&](auto term) {
        float half[H];
#pragma unroll
        for (int h = 0; h < H; ++h) {
            float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
            for (int i = h * PER; i < (h + 1) * PER; ++i)
                if (c.real[i]) {
                    const float4 t = term(v[i]);
                    s = make_float4(s.x + t.x, s.y + t.y, s.z + t.z, s.w + t.w);
                }
            half[h] = wave_sum_ascending((s.x + s.y) + (s.z + s.w));
        }
        return PAIR ? half[0] + half[H - 1] : half[0];
    };
    const float cols_f = static_cast<float>(c.cols);
    const float mean = total([](const float4 &t) { return t; }) / cols_f;
    const float var = total([&](const float4 &t) {
        const float p = t.x - mean, q = t.y - mean, r = t.z - mean, s = t.w - mean;
        return make_float4(p * p, q * q, r * r, s * s);
    }) / cols_f;
    const float rstd = 1.0f / sqrtf(var + eps);
    float am = 0.0f;
#pragma unroll
    for (int i = 0; i < RC; ++i) {
        if (!c.real[i]) continue;
        v[i] = make_float4((v[i].x - mean) * rstd * a.g[i].x + a.b[i].x, (v[i].y - mean) * rstd * a.g[i].y + a.b[i].y,
                           (v[i].z - mean) * rstd * a.g[i].z + a.b[i].z, (v[i].w - mean) * rstd * a.g[i].w + a.b[i].w);
        am = fmaxf(fmaxf(am, fmaxf(fabsf(v[i].x), fabsf(v[i].y))), fmaxf(fabsf(v[i].z), fabsf(v[i].w)));
    }
    am = wave_max(am);
    float scale = am < FLT_EPSILON ? 1.0f : am / 127.0f;
    if (!(fabsf(am) <= FLT_MAX)) scale = NAN;
    const float inv = recip_for_div(scale);
#pragma unroll
    for (int i = 0; i < RC; ++i)
        if (c.real[i])
            q[i] = pack4(quantize_int_sym<EVEN>(v[i].x, scale, inv), quantize_int_sym<EVEN>(v[i].y, scale, inv),
                         quantize_int_sym<EVEN>(v[i].z, scale, inv), quantize_int_sym<EVEN>(v[i].w, scale, inv));
    return scale;
}

// Per-token int8 of the row: its codes in q, its scale returned (NaN, with zero codes, for a row whose range is not finite, so
// that every output of the row is NaN).
template <bool EVEN, int RC>
__device__ __forceinline__ float row_range_quantize(const float4 (&v)[RC], const PanelColumns<RC, false> &c, uint32_t (&q)[RC]) {
    float mn = INFINITY, mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < RC; ++i)
        if (c.real[i]) {
            mn = fminf(mn, fminf(fminf(v[i].x, v[i].y), fminf(v[i].z, v[i].w)));
            mx = fmaxf(mx, fmaxf(fmaxf(v[i].x, v[i].y), fmaxf(v[i].z, v[i].w)));
        }
    float scale;
    int zp;
    const bool good =
        params_from_minmax(wave_min(mn), wave_max(mx), HIPQ_PARAMS_SYMMETRIC, -128, 127, &scale, &zp) == HIPQ_SUCCESS;
    const float inv = recip_for_div(scale);
#pragma unroll
    for (int i = 0; i < RC; ++i)
        q[i] = good ? pack4(quantize_int_sym<EVEN>(v[i].x, scale, inv), quantize_int_sym<EVEN>(v[i].y, scale, inv),
                            quantize_int_sym<EVEN>(v[i].z, scale, inv), quantize_int_sym<EVEN>(v[i].w, scale, inv))
                    : 0u;
    return good ? scale : NAN;
}

}  // namespace hipq
