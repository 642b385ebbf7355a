// Quantized Linear of small sizes in one launch: fp32 rows -> int8 -> product -> fp32.
//
// A quantizer and a product, each a launch and a few dependent trips to memory, are 4 us apiece whatever they move, one behind the
// other.  Here a workgroup owns 16 rows x 32 columns and quantizes its rows itself: sixteen waves, a row each, the codes to LDS
// in fragment order, then K split between the waves, partial sums through LDS.  The weights are requested in front of the rows.
// The row operation is repeated by every workgroup of a row tile, and a tensor's range is found by every workgroup for itself, so
// this is for few workgroups on short rows.  Products are v_mfma_i32_16x16x64_i8: operands, a lane's 16 bytes are of row or column
// lane % 16 and quarter lane / 16 of 64 bytes of K; results, column lane % 16 and rows 4 (lane / 16) + 0 .. 3.
#include "hipq_gemm_split.h"
#include "hipq_internal.h"

namespace hipq {
namespace {

constexpr int kSmallRows = 16, kSmallWaves = 16;

struct LinearSmall {
    const float *x;
    const int8_t *w;
    const float *w_scales, *bias;
    float *out;
    float scale;  // static
    int range, m, n, k, aligned;
};

// The row's floats 4 (lane + 64 i) .. + 3; NaN past its end.
template <int RC>
__device__ __forceinline__ void load_row(const float *row, int lane, int K, AnyFloat4 (&v)[RC]) {
#pragma unroll
    for (int i = 0; i < RC; ++i) {
        const int c = 4 * (lane + kWave * i);
        if (c + 4 <= K) {
            v[i] = *reinterpret_cast<const AnyFloat4 *>(row + c);
        } else {
            const float none = __builtin_nanf("");
            v[i] = AnyFloat4{c < K ? row[c] : none, c + 1 < K ? row[c + 1] : none, c + 2 < K ? row[c + 2] : none, none};
        }
    }
}

__device__ __forceinline__ void widen(float &mn, float &mx, const AnyFloat4 &v) {
    mn = fminf(mn, fminf(fminf(v.x, v.y), fminf(v.z, v.w)));
    mx = fmaxf(mx, fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)));
}

// RC float4 a lane hold a row of up to 256 RC floats; ROWS: weights as rows of K bytes (K >= 16), else packed.
template <int RC, bool ROWS, bool DIV, bool EVEN>
__global__ __launch_bounds__(1024) void linear_small_kernel(LinearSmall p) {
    constexpr int kPiece = kSmallRows + 1;  // (a piece of padding: the lanes of a store hit all banks)
    constexpr int STEPS = (RC * 4 + kSmallWaves - 1) / kSmallWaves;
    constexpr bool EARLY = !(ROWS && RC > 4);  // (unaligned pieces in flight take too many registers beside long rows)
    __shared__ __attribute__((aligned(16))) v4i codes[RC * 16 * kPiece];  // [16 bytes of K][row]
    __shared__ __attribute__((aligned(16))) v4i part[kSmallWaves][2][kWave];
    __shared__ float row_scale[kSmallRows], wave_mn[kSmallWaves], wave_mx[kSmallWaves];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int M = p.m, N = p.n, K = p.k;
    const int row0 = static_cast<int>(blockIdx.y) * kSmallRows, col0 = static_cast<int>(blockIdx.x) * 32;
    const int KB = static_cast<int>(packed_k_blocks(K)), quads = ROWS ? (K + 63) / 64 : KB / 2;  // 64 bytes of K each
    const float *xr = p.x + size_t(row0 + wave < M ? row0 + wave : M - 1) * K;

    v4i fw[STEPS][2];
    auto weights = [&](auto use) {
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const int q = wave + kSmallWaves * s;
            if (q >= quads) break;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                if constexpr (ROWS) {
                    const int n = col0 + 16 * c + lane % 16, k = 64 * q + 16 * (lane / 16);
                    const int8_t *row = p.w + size_t(n < N ? n : N - 1) * K;
                    if (p.aligned) {
                        use(s, c, [=] { return k < K ? *reinterpret_cast<const v4i *>(row + k) : v4i{0, 0, 0, 0}; });
                    } else {
                        TailPiece t;
                        t.load(RowStart(row), k < K ? k : K, K);
                        use(s, c, [=] { return t.get(); });
                    }
                } else {
                    const int8_t *from = p.w + (size_t(col0 / 32) * KB + 2 * q) * 1024 + (lane / 16) * 512 + (16 * c + lane % 16) * 16;
                    use(s, c, [=] { return *reinterpret_cast<const v4i *>(from); });
                }
            }
        }
    };
    auto fetch = [&] { weights([&](int s, int c, auto value) { fw[s][c] = value(); }); };
    if constexpr (EARLY) fetch();
    // wave c finishes columns col0 + 16 c + 0 .. 15
    const int n = col0 + 16 * (wave % 2) + lane % 16, nc = n < N ? n : N - 1, mine = 4 * (lane / 16);
    float sw = 0.0f, bias = 0.0f;
    if (wave < 2) {
        sw = p.w_scales[nc];
        if (p.bias) bias = p.bias[nc];
    }
    AnyFloat4 v[RC];
    load_row<RC>(xr, lane, K, v);
    float scale = p.scale;
    bool good = true;
    if (p.range != LINEAR_STATIC) {
        float mn = INFINITY, mx = -INFINITY;
        if (p.range == LINEAR_PER_TOKEN) {
#pragma unroll
            for (int i = 0; i < RC; ++i) widen(mn, mx, v[i]);
            mn = wave_min(mn);
            mx = wave_max(mx);
        } else {
            const int total = M * K, whole = total / 4;
#pragma unroll 4
            for (int f = threadIdx.x; f < whole; f += kSmallWaves * kWave) widen(mn, mx, reinterpret_cast<const AnyFloat4 *>(p.x)[f]);
            if (threadIdx.x < static_cast<unsigned>(total - 4 * whole)) {
                const float e = p.x[4 * whole + threadIdx.x];
                mn = fminf(mn, e);
                mx = fmaxf(mx, e);
            }
            mn = wave_min(mn);
            mx = wave_max(mx);
            if (lane == 0) {
                wave_mn[wave] = mn;
                wave_mx[wave] = mx;
            }
            __syncthreads();
#pragma unroll
            for (int w = 0; w < kSmallWaves; ++w) {
                mn = fminf(mn, wave_mn[w]);
                mx = fmaxf(mx, wave_mx[w]);
            }
        }
        int zp;
        good = params_from_minmax(mn, mx, HIPQ_PARAMS_SYMMETRIC, -128, 127, &scale, &zp) == HIPQ_SUCCESS;
    }
    // A range that is not finite: NaN scale and zero codes, so that every output is NaN.
    if (lane == 0) row_scale[wave] = good ? scale : NAN;
    const float inv = DIV ? recip_for_div(scale) : 1.0f / scale;
    // (quantize_int, with the choice of its division made once per row)
    auto row_codes = [&](auto by_reciprocal) {
        auto code = [&](float x) {
            float t;
            if constexpr (!DIV) {
                t = x * inv;
            } else if constexpr (decltype(by_reciprocal)::value) {
                const float q0 = x * inv, q1 = fmaf(fmaf(-q0, scale, x), inv, q0);
                t = q1 == q1 ? q1 : q0;
            } else {
                t = x / scale;
            }
            return min(max(cvt_i32_sat(round_mode<EVEN>(t)), -128), 127);
        };
        uint32_t *dword = reinterpret_cast<uint32_t *>(codes);
#pragma unroll
        for (int i = 0; i < RC; ++i) {
            const int f = lane + kWave * i;  // (past the row, up to the last quad: NaN, code 0)
            if (f < quads * 16)
                dword[(f / 4 * kPiece + wave) * 4 + f % 4] = good ? pack4(code(v[i].x), code(v[i].y), code(v[i].z), code(v[i].w)) : 0u;
        }
    };
    if (!DIV || inv != 0.0f)
        row_codes(std::true_type{});
    else
        row_codes(std::false_type{});
    if constexpr (!EARLY) fetch();
    __syncthreads();
    v4i acc[2] = {v4i{0, 0, 0, 0}, v4i{0, 0, 0, 0}};
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        const int q = wave + kSmallWaves * s;
        if (q >= quads) break;
        const v4i fa = codes[(4 * q + lane / 16) * kPiece + lane % 16];
#pragma unroll
        for (int c = 0; c < 2; ++c) acc[c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa, fw[s][c], acc[c], 0, 0, 0);
    }
    const int active = quads < kSmallWaves ? quads : kSmallWaves;  // waves with a share of K
    if (wave < active) {
#pragma unroll
        for (int c = 0; c < 2; ++c) part[wave][c][lane] = acc[c];
    }
    __syncthreads();
    if (wave >= 2 || n >= N) return;
    v4i sum = part[0][wave][lane];
#pragma unroll
    for (int w = 1; w < kSmallWaves; ++w)
        if (w < active) sum += part[w][wave][lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = row0 + mine + i;
        if (m >= M) break;
        float o = static_cast<float>(sum[i]) * (row_scale[mine + i] * sw);
        if (p.bias) o = o + bias;
        p.out[size_t(m) * N + n] = o;
    }
}

template <int RC, bool ROWS>
void launch(hipq_ctx *ctx, const LinearSmall &p, bool div, bool even) {
    const dim3 grid(static_cast<unsigned>((p.n + 31) / 32), static_cast<unsigned>((p.m + kSmallRows - 1) / kSmallRows));
#define HIPQ_SMALL(D, E) hipLaunchKernelGGL((linear_small_kernel<RC, ROWS, D, E>), grid, dim3(1024), 0, ctx->stream, p)
    if (div && even)
        HIPQ_SMALL(true, true);
    else if (div)
        HIPQ_SMALL(true, false);
    else if (even)
        HIPQ_SMALL(false, true);
    else
        HIPQ_SMALL(false, false);
#undef HIPQ_SMALL
}

}  // namespace

// The lines, by what both take inside a graph (us, quantizer and product / this); launched one by one the two take 8.4 and more.
//   static scale, up to two workgroups per compute unit: K <= 1024 2 x 64 x 384 4.9 / 3.5, 104 x 128 x 128 5.1 / 3.4, 159 x 384 x
//     832 5.6 / 4.6, 1 x 1984 x 64 4.9 / 3.3, 724 x 254 x 64 5.2 / 4.5, 3 x 15936 x 769 6.6 / 6.0, three: 5082 x 64 x 384 6.8 / 6.5; packed
//     weights up to K = 2048, one: 6 x 64 x 1600 5.8 / 5.5, 298 x 64 x 1765 6.4 / 5.8, two: 492 x 323 x 1400 7.3 / 9.3; rows: 24 x 896 x
//     1633 6.1 / 6.7
//   per token, up to one per compute unit, K <= 1024: 22 x 104 x 64 5.1 / 4.1, 294 x 256 x 64 6.0 / 4.3, 46 x 1280 x 832 6.2 / 5.7; two:
//     447 x 320 x 896 6.7 / 7.7; longer rows: 28 x 2240 x 1600 6.5 / 7.5, 75 x 128 x 1242 6.8 / 7.4
//   per tensor, the same, of up to 64 Ki floats, which every workgroup reads: 2 x 64 x 320 6.9 / 4.2, 69 x 256 x 192 7.6 / 4.8, 145 x
//     128 x 256 7.3 / 5.3, 17 x 3328 x 1716 8.5 / 8.2, but 152 x 64 x 645 8.4 / 8.4, 309 x 64 x 832 8.2 / 12.8
bool linear_small(hipq_ctx *ctx, LinearRange range, const float *x, float scale, const int8_t *w, bool w_rows, const float *w_scales,
                  const float *bias, size_t m, size_t n, size_t k, int32_t mode, float *out, int32_t *rc) {
    if (ctx->gemm_variant != 0 || ctx->trace || (w_rows && k < 16)) return false;
    if (range != LINEAR_PER_TOKEN && (mode & ~(HIPQ_ROUND_HALF_EVEN | HIPQ_FORM_DIV))) return false;  // (the quantizer says so)
    if (range == LINEAR_STATIC && !(scale > 0.0f)) return false;
    const bool longer = k > 1024;
    if (k > 2048 || (longer && (range == LINEAR_PER_TOKEN || (range == LINEAR_STATIC && w_rows)))) return false;
    const size_t most = size_t(ctx->num_cus) * (range == LINEAR_STATIC && !longer ? 2 : 1);
    if (m > most * kSmallRows || n > most * 32 || (m + kSmallRows - 1) / kSmallRows * ((n + 31) / 32) > most) return false;
    if (range == LINEAR_PER_TENSOR && m * k > 65536) return false;
    // A result over its input (an in-place call): a workgroup would store into rows that others have not read.  The quantizer has read
    // all of x before the product stores anything.
    if (memory_meets(x, m * k * sizeof(float), out, m * n * sizeof(float))) return false;
    const LinearSmall p{x, w, w_scales, bias, out, scale, range, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k),
                        k % 16 == 0 && (reinterpret_cast<uintptr_t>(w) & 15u) == 0};
    const bool div = range == LINEAR_PER_TOKEN || (mode & HIPQ_FORM_DIV), even = (mode & HIPQ_ROUND_HALF_EVEN) != 0;
    if (k <= 1024 && w_rows)
        launch<4, true>(ctx, p, div, even);
    else if (k <= 1024)
        launch<4, false>(ctx, p, div, even);
    else if (w_rows)
        launch<8, true>(ctx, p, div, even);
    else
        launch<8, false>(ctx, p, div, even);
    *rc = check_launch("linear (small)");
    return true;
}

}  // namespace hipq
