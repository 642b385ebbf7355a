// Per-token int8 quantizer into the fragment-packed operand layout of the packed GEMM
// ([row block of 32][k block of 32 bytes][1 KiB]; lane l of a fragment = row l % 32, bytes 16 * (l / 32) .. +15).
//
// A workgroup owns ROWS rows, LPR lanes each; a lane holds VPT float4 of its row between the range and the codes, so rows
// are read once.  The 16 bytes that a row has in a fragment lie 512 bytes from its next ones: a row on its own writes
// pieces of lines that other workgroups, mostly on other dies, write the rest of.  The codes therefore cross LDS and leave
// as 16 bytes a lane, the ROWS rows side by side.  Rows at any alignment of a float; what pads the operand (rows to a
// multiple of 32, K to one of 128) is written as zeros.
#pragma once

#include "hipq_internal.h"
#include "hipq_math.h"

namespace hipq {

struct __attribute__((packed, aligned(4))) Floats4 {
    float v[4];
};

// tanh-form GELU, crates/torsh-nn/src/layers/activation/modern.rs:124-136:
//   0.5 * x * (1 + tanh(u)),  u = sqrt(2/pi) * (x + 0.044715 x^3).
// Evaluated as x / (1 + exp(-2u)), which is the same function (1 + tanh(u) = 2 / (1 + exp(-2u)))
// without the cancellation of 1 + tanh(u) for negative x, and costs one v_exp_f32 and one
// v_rcp_f32 instead of a tanhf call: the fused GELU + quantize kernel was bound by tanhf, not by
// HBM.  Against the reference's evaluation order in f32 the difference stays below 2e-6
// relative + 1e-7 absolute (the reference form itself carries up to |x| * 3e-8 of cancellation
// error).
// -2u * log2(e) = x * (K + K*c*x^2) with K = -2*log2(e)*sqrt(2/pi): one multiply, one fused
// multiply-add, one multiply (this function is compared at a tolerance, so the contraction is
// allowed here).  No clamp of the exponent: exp2 saturates to inf / 0, and rcp(1 + inf) = 0,
// rcp(1 + 0) = 1 give the right limits x * 0 and x.
__device__ __forceinline__ float gelu_tanh(float x) {
    constexpr float K = -2.8853900817779268f * 0.7978845608028654f;
    const float arg = x * fmaf(x * x, K * 0.044715f, K);
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(arg));
}

// GELU: of the activated row, with the scale of the row kernels (a row of NaN elements has the maximum 0).
template <int LPR, int ROWS, int VPT, bool EVEN, bool GELU>
__global__ __launch_bounds__(LPR *ROWS) void quantize_rows_packed_kernel(const float *__restrict__ x, unsigned rows, unsigned cols,
                                                                         size_t ld, int8_t *__restrict__ out,
                                                                         float *__restrict__ out_scales, unsigned dies) {
    static_assert(LPR % kWave == 0 && 32 % ROWS == 0, "whole waves per row, whole workgroups per row block");
    constexpr int kThreads = LPR * ROWS, kWavesPerRow = LPR / kWave, kRun = ROWS > 1 ? ROWS + 1 : 1;
    constexpr unsigned kPerBlock = 32 / ROWS;
    __shared__ float lds_mn[kThreads / kWave], lds_mx[kThreads / kWave];
    __shared__ __attribute__((aligned(16))) uint32_t codes[VPT * LPR / 4][kRun][4];  // [16 bytes of K][row][dword]
    // The workgroups of a row block on one die (dies = 8), so that its L2 joins the pieces of a line.
    const unsigned in_die = blockIdx.x / dies;
    const unsigned block = in_die / kPerBlock * dies + blockIdx.x % dies;
    if (block >= (rows + 31) / 32) return;
    const unsigned row0 = block * 32 + in_die % kPerBlock * ROWS;
    const unsigned sub = threadIdx.x / LPR, lane = threadIdx.x % LPR, row = row0 + sub;
    const bool active = row < rows;
    const float *xr = x + (active ? row : 0) * ld;
    const unsigned mine = active ? cols : 0;
    Floats4 v[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const unsigned c = 4 * (lane + unsigned(i) * LPR);
        // past the end: neither the minimum nor the maximum changes, and the code is 0
#pragma unroll
        for (int j = 0; j < 4; ++j) v[i].v[j] = __builtin_nanf("");
        if (c + 4 <= mine) {
            v[i] = *reinterpret_cast<const Floats4 *>(xr + c);
        } else {
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (c + j < mine) v[i].v[j] = xr[c + j];
        }
    }
    if constexpr (GELU) {
#pragma unroll
        for (int i = 0; i < VPT; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[i].v[j] = gelu_tanh(v[i].v[j]);
    }
    float mn = GELU ? 0.0f : INFINITY, mx = GELU ? 0.0f : -INFINITY;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        mn = fminf(mn, fminf(fminf(v[i].v[0], v[i].v[1]), fminf(v[i].v[2], v[i].v[3])));
        mx = fmaxf(mx, fmaxf(fmaxf(v[i].v[0], v[i].v[1]), fmaxf(v[i].v[2], v[i].v[3])));
    }
    mn = wave_min(mn);
    mx = wave_max(mx);
    if constexpr (kWavesPerRow > 1) {
        if (threadIdx.x % kWave == 0) {
            lds_mn[threadIdx.x / kWave] = mn;
            lds_mx[threadIdx.x / kWave] = mx;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kWavesPerRow; ++w) {
            mn = fminf(mn, lds_mn[sub * kWavesPerRow + w]);
            mx = fmaxf(mx, lds_mx[sub * kWavesPerRow + w]);
        }
    }
    float scale;
    [[maybe_unused]] int zp;
    // A row whose range is not finite gets a NaN scale and zero codes, so that every output of it is NaN.
    bool good;
    if constexpr (GELU) {
        const float am = fmaxf(fabsf(mn), fabsf(mx));
        scale = am < FLT_EPSILON ? 1.0f : am / 127.0f;
        good = am <= FLT_MAX;
    } else {
        good = params_from_minmax(mn, mx, HIPQ_PARAMS_SYMMETRIC, -128, 127, &scale, &zp) == HIPQ_SUCCESS;
    }
    if (active && lane == 0) out_scales[row] = good ? scale : __builtin_nanf("");
    const float inv = recip_for_div(scale);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const unsigned at = lane + unsigned(i) * LPR;
        const uint32_t q = pack4(quantize_int_sym<EVEN>(v[i].v[0], scale, inv), quantize_int_sym<EVEN>(v[i].v[1], scale, inv),
                                 quantize_int_sym<EVEN>(v[i].v[2], scale, inv), quantize_int_sym<EVEN>(v[i].v[3], scale, inv));
        codes[at / 4][sub][at % 4] = good ? q : 0u;
    }
    __syncthreads();
    const unsigned pieces = (cols + 127) / 128 * 8;  // of 16 bytes of K
    int8_t *base = out + size_t(block) * pieces * 512 + row0 % 32 * 16;
    for (unsigned e = threadIdx.x; e < pieces * ROWS; e += kThreads) {
        const unsigned g = e / ROWS, r = e % ROWS;
        *reinterpret_cast<uint4 *>(base + size_t(g) * 512 + r * 16) = *reinterpret_cast<const uint4 *>(codes[g][r]);
    }
}

// The longest rows that a workgroup's registers hold (the longest form).
constexpr size_t kRowsPackedMaxCols = 16384;

// Four float4 a lane while the device's lanes hold the whole matrix like that at once (2048 lanes a compute unit), else eight
// on half the lanes.  us, four / eight, inputs from memory: 1024 x 4096 6.7 / 7.4, 2048 x 4096 9.8 / 10.7, 4096 x 4096 17.3 /
// 16.4 (a row per workgroup of 256, its codes stored where they lie: 28.3), 4096 x 11008 42.3 / 35.3 (60.3), 1000 x 11008
// 15.3 / 13.6 (18.1).  Rows of up to 2048 floats: four, 8192 x 2048 16.0 / 17.9 (26.8).  Rows that start at an odd float lose
// nothing: 4096 x 4095 16.8 (49.9).
// Few rows want a workgroup each: 64 x 8000 4.7, two side by side 4.9 (6.5); 16 x 11008 5.0 (6.8); 16 x 3072 4.4, four side by side
// 5.1 (4.6); 1 x 2048 4.1, 4.4 (4.2); as many as compute units they are even, 300 x 2100 5.3, 5.3 (5.3).  Short rows want one
// float4 a lane, the others are work for nothing: 6852 x 128 5.4, four 6.6 (5.4); 2667 x 54 4.3, 4.9 (4.5).
// GELU is twice the vector work: a row per workgroup until there are four per compute unit (640 tokens at d_ff 3072).
template <bool EVEN, bool GELU = false>
static void launch_quantize_rows_packed(hipq_ctx *ctx, const float *x, size_t rows, size_t cols, size_t ld, int8_t *out,
                                        float *out_scales) {
    const size_t row_blocks = (rows + 31) / 32;
    const unsigned dies = row_blocks >= 16 ? 8 : 1;  // (fewer blocks: every die gets workgroups of each)
    const bool many = rows * cols > size_t(ctx->num_cus) * 2048 * 16;
    const bool few = rows < size_t(ctx->num_cus) * (GELU ? 4 : 1);
#define HIPQ_ROWS_PACKED(LPR, ROWS, VPT)                                                                                     \
    hipLaunchKernelGGL((quantize_rows_packed_kernel<LPR, ROWS, VPT, EVEN, GELU>),                                            \
                       dim3(static_cast<unsigned>((row_blocks + dies - 1) / dies * dies * (32 / ROWS))), dim3(LPR * ROWS), 0, \
                       ctx->stream, x, static_cast<unsigned>(rows), static_cast<unsigned>(cols), ld, out, out_scales, dies)
    if (cols <= 256)
        HIPQ_ROWS_PACKED(64, 4, 1);
    else if (cols <= 1024)
        HIPQ_ROWS_PACKED(64, 4, 4);
    else if (!GELU && cols <= 2048 && few)
        HIPQ_ROWS_PACKED(256, 1, 2);
    else if (cols <= 2048)
        HIPQ_ROWS_PACKED(128, 4, 4);
    else if (cols <= 4096 && few)
        HIPQ_ROWS_PACKED(256, 1, 4);
    else if (cols <= 4096 && !many)
        HIPQ_ROWS_PACKED(256, 4, 4);
    else if (cols <= 4096)
        HIPQ_ROWS_PACKED(128, 4, 8);
    else if (cols <= 8192 && !many)
        HIPQ_ROWS_PACKED(512, 1, 4);
    else if (cols <= 8192)
        HIPQ_ROWS_PACKED(256, 2, 8);
    else if (!many)
        HIPQ_ROWS_PACKED(1024, 1, 4);
    else
        HIPQ_ROWS_PACKED(512, 1, 8);
#undef HIPQ_ROWS_PACKED
}

}  // namespace hipq
