// Linear of few tokens with the row operation that makes its int8 activations in front: x (fp32 rows) -> LayerNorm and
// per-token int8, or per-token int8 alone -> product with packed weights -> fp32.
//
// With a few dozen tokens the quantizing kernel and the product are a launch and a few dependent trips to memory each, 3.5 to
// 4 us apiece whatever they move.  Here a workgroup owns 16 rows x 32 CB columns and runs the row operation on its rows itself:
// sixteen waves, a row each, the codes to LDS in fragment order, then K split between the waves, partial sums through LDS.
// The weights are requested behind the rows and arrive meanwhile.  The row operation is repeated by every workgroup of a
// row block, so this is for as many workgroups as the compute units take at once.
#include "hipq_internal.h"
#include "hipq_panel_norm.h"

namespace hipq {

using v4i = __attribute__((__vector_size__(4 * sizeof(int)))) int;
using v16i = __attribute__((__vector_size__(16 * sizeof(int)))) int;

constexpr int kRowOpBlocks = 3;  // float4 a lane per row

template <bool NORM, int CB, bool EVEN>
__global__ __launch_bounds__(1024) void row_op_split_kernel(RowOpLinear p) {
    constexpr int RC = kRowOpBlocks, WK = 16, ROWS = 16, STEPS = (RC * 8 + WK - 1) / WK;
    constexpr int kPiece = ROWS + 1;  // 16-byte pieces of a half k block, one of padding: the lanes of a store hit all banks
    __shared__ __attribute__((aligned(16))) v4i codes[RC * 8 * 2 * kPiece];  // [k block][half][row]
    __shared__ __attribute__((aligned(16))) v4i part[WK][2 * CB][kWave];
    __shared__ float row_scale[ROWS];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int M = static_cast<int>(p.rows), N = static_cast<int>(p.n), KB = static_cast<int>(p.k / 32);
    const int row0 = static_cast<int>(blockIdx.y) * ROWS, col0 = static_cast<int>(blockIdx.x) * 32 * CB;
    const PanelColumns<RC, false> c(lane, KB);
    // the wave's row (rows past the last are computed and discarded)
    const float *xr = p.x + size_t(row0 + wave < M ? row0 + wave : M - 1) * p.ld;
    float4 v[RC];
#pragma unroll
    for (int i = 0; i < RC; ++i) v[i] = c.real[i] ? *reinterpret_cast<const float4 *>(xr + c.at(i)) : float4{};
    const PanelAffine<RC> affine(c, NORM ? p.gamma : nullptr, NORM ? p.beta : nullptr);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(p.w), 0, 0x7fffffff, 0x00020000);
    v4i fw[STEPS][CB];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        const int kb = wave + WK * s;
#pragma unroll
        for (int j = 0; j < CB; ++j)  // (k blocks past the last: zeros, no memory access)
            fw[s][j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, kb < KB ? lane * 16 : 0x7fffffff,
                                                                                     kb < KB ? ((col0 / 32 + j) * KB + kb) * 1024 : 0, 0));
    }
    // Wave 2 j + g finishes rows 8 g + 4 (lane / 32) + 0 .. 3 of column block j.
    const int n = col0 + 32 * (wave / 2) + lane % 32, mine = 8 * (wave % 2) + 4 * (lane / 32);
    float sw = 0.0f, bias = 0.0f, residual[4];
    if (wave < 2 * CB) {
        sw = p.w_scales[n];
        if (p.bias) bias = p.bias[n];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = row0 + mine + i;
            residual[i] = p.residual ? p.residual[size_t(m < M ? m : M - 1) * N + n] : 0.0f;
        }
    }
    uint32_t q[RC];
    float scale;
    if constexpr (NORM) {
        scale = panel_norm_quantize<EVEN>(v, c, affine, p.eps, q);
    } else {
        scale = row_range_quantize<EVEN>(v, c, q);
    }
    if (lane == 0) row_scale[wave] = scale;
    uint32_t *dword = reinterpret_cast<uint32_t *>(codes);
#pragma unroll
    for (int i = 0; i < RC; ++i)
        if (c.real[i]) dword[((c.block[i] * 2 + c.part / 4) * kPiece + wave) * 4 + c.part % 4] = q[i];
    __syncthreads();
    v16i acc[CB];
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        const int kb = wave + WK * s;
        if (kb >= KB) break;
        // (operand rows 16 .. 31 repeat 0 .. 15; their results are not looked at)
        const v4i fa = codes[(kb * 2 + lane / 32) * kPiece + lane % ROWS];
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fw[s][j], acc[j], 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
        for (int g = 0; g < 2; ++g)
            part[wave][2 * j + g][lane] = v4i{acc[j][4 * g], acc[j][4 * g + 1], acc[j][4 * g + 2], acc[j][4 * g + 3]};
    __syncthreads();
    if (wave >= 2 * CB) return;
    v4i sum = part[0][wave][lane];
#pragma unroll
    for (int w = 1; w < WK; ++w) sum += part[w][wave][lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = row0 + mine + i;
        if (m >= M) continue;
        float o = static_cast<float>(sum[i]) * (row_scale[mine + i] * sw);
        if (p.bias) o = o + bias;
        if (p.residual) o = o + residual[i];
        p.out[size_t(m) * N + n] = o;
    }
}

// Rows of up to 768 floats (three float4 a lane) and no more workgroups than compute units, two column blocks each where one
// makes more.  Twelve layers, us, separate kernels / this: d 768, d_ff 3072 1 token 322 / 286, 16 335 / 308, 77 365 / 333, 128
// 368 / 350, 200 393 / 381, 300 423 / 421; d 128, d_ff 512 200 tokens 316 / 277; d 512 100 tokens 323 / 310.  Two workgroups
// per compute unit: d 768 128 tokens 439, 200 514.  Rows of 1024 floats: one wave holds too much, 77 tokens 381 / 491.
bool row_op_linear_fits(const hipq_ctx *ctx, const float *x, size_t rows, size_t n, size_t k, PanelFold fold) {
    return !fold.pair && fold.wave_blocks == kRowOpBlocks && k % 128 == 0 && k <= kRowOpBlocks * 256 && n % 64 == 0 &&
           (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && (rows + 15) / 16 * (n / 64) <= size_t(ctx->num_cus);
}

int32_t row_op_linear(hipq_ctx *ctx, const RowOpLinear &p, int32_t mode) {
    const size_t row_blocks = (p.rows + 15) / 16;
    const bool two = row_blocks * (p.n / 32) > size_t(ctx->num_cus), even = (mode & HIPQ_ROUND_HALF_EVEN) != 0;
    const dim3 grid(static_cast<unsigned>(p.n / (two ? 64 : 32)), static_cast<unsigned>(row_blocks));
#define HIPQ_ROW_OP(NORM, CB, E) hipLaunchKernelGGL((row_op_split_kernel<NORM, CB, E>), grid, dim3(1024), 0, ctx->stream, p)
#define HIPQ_ROW_OP_FORM(NORM)                         \
    do {                                               \
        if (two && even) HIPQ_ROW_OP(NORM, 2, true);   \
        else if (two) HIPQ_ROW_OP(NORM, 2, false);     \
        else if (even) HIPQ_ROW_OP(NORM, 1, true);     \
        else HIPQ_ROW_OP(NORM, 1, false);              \
    } while (0)
    if (p.norm)
        HIPQ_ROW_OP_FORM(true);
    else
        HIPQ_ROW_OP_FORM(false);
#undef HIPQ_ROW_OP_FORM
#undef HIPQ_ROW_OP
    return check_launch("row operation + linear");
}

}  // namespace hipq
