// int8 GEMM on row-major operands of any K >= 16 and alignment, few tiles: K split between the waves of a workgroup.
//
// A product of few tiles is latency: a tiled kernel walks K with one or two K-tiles in flight and leaves compute units
// idle.  Here a workgroup of WK waves owns a tile of 16 FM x 16 FN outputs, wave w takes the steps w, w + WK, ... of
// 64 P bytes of K and loads its rows' pieces straight into the operand registers of v_mfma_i32_16x16x64_i8 (no LDS:
// nothing is shared between waves that split K), a step in flight per wave, and the partial sums meet in LDS once.  A lane
// takes 16 P consecutive bytes of its row per step (the sums do not care which bytes of K share an MFMA, as long as both
// operands agree), which is what makes odd rows affordable: they need one dword more per P pieces.
//
// Bound by the vector-memory path (a compute unit takes ~28 operand bytes per ns with the shift, ~36 without) behind
// ~3.3 us of launch, first round trip and the meeting of the partial sums.  300 x 1000 x 1001 11.7 -> 6.6 us, x 1008 8.0 ->
// 5.6, 64 x 4096 x 4097 26.0 -> 12.7.  P = 1 instead of 2: 8.0 at 1001; loads at the byte address: 10.2.
#pragma once

#include "hipq_gemm_kernels.h"

namespace hipq {

// Scales, biases and residuals of four consecutive outputs of a row, requested ahead of the K loop.
struct EpilogueOperands {
    float sw[4], bias[4], residual[4], sa;
};
template <int EPI>
__device__ __forceinline__ EpilogueOperands load_epilogue_operands(const GemmEpilogue &ep, int m, int n, int M, int N) {
    EpilogueOperands o{};
    if constexpr (EPI != EPI_I32) {
        const int mc = m < M ? m : M - 1;
        o.sa = ep.sa_per_row ? ep.sa[mc] : ep.sa[0];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int nc = n + i < N ? n + i : N - 1;
            o.sw[i] = ep.sw[nc];
            if (ep.bias) o.bias[i] = ep.bias[nc];
            if (ep.residual) o.residual[i] = ep.residual[size_t(mc) * N + nc];
        }
    }
    return o;
}

template <int EPI, bool EVEN>
__device__ __forceinline__ void epilogue_store4_loaded(const GemmEpilogue &ep, const EpilogueOperands &o, int m, int n, int M,
                                                       int N, v4i acc) {
    if (m >= M || n >= N) return;
    const size_t off = size_t(m) * N + n;
    constexpr unsigned kAlignMask = (EPI == EPI_I8) ? 3u : 15u;
    const bool vec = (N % 4 == 0) && ((reinterpret_cast<uintptr_t>(ep.out) & kAlignMask) == 0);
    if constexpr (EPI == EPI_I32) {
        int32_t *out = static_cast<int32_t *>(ep.out);
        if (vec) {
            *reinterpret_cast<v4i *>(out + off) = acc;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (n + i < N) out[off + i] = acc[i];
        }
    } else {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float s = o.sa * o.sw[i];
            v[i] = static_cast<float>(acc[i]) * s;
            if (ep.bias) v[i] = v[i] + o.bias[i];
            if (ep.residual) v[i] = v[i] + o.residual[i];
        }
        if constexpr (EPI == EPI_F32) {
            float *out = static_cast<float *>(ep.out);
            if (vec) {
                *reinterpret_cast<float4 *>(out + off) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < N) out[off + i] = v[i];
            }
        } else {
            int8_t *out = static_cast<int8_t *>(ep.out);
            int q[4];
            const float zpf = static_cast<float>(ep.zp_out);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                q[i] = to_int_nan0(clamp_keep_nan(round_mode<EVEN>(div_rn(v[i], ep.s_out, ep.s_out_inv)) + zpf, -128.0f, 127.0f));
            if (vec) {
                *reinterpret_cast<uint32_t *>(out + off) = pack4(q[0], q[1], q[2], q[3]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < N) out[off + i] = static_cast<int8_t>(q[i]);
            }
        }
    }
}

// 16 bytes of a row at any alignment as whole dwords: a load whose lanes are not dword aligned runs at a quarter of the
// rate or less (M = 300, N = 1000 at K = 1001 / 1002 / 1004 / 1008: 10.2 / 10.2 / 5.4 / 5.1 us).  `raw` holds the aligned
// dwords that the piece touches - the fifth only where it touches it - and get() shifts them into place, so that a batch
// of loads is in flight before the first shift.  Nothing outside the dwords that hold bytes of the piece is read.
struct __attribute__((packed, aligned(4))) Dwords16 {
    v4i v;
};
template <int P>
struct ShiftedPieces {  // P pieces of 16 bytes, consecutive
    v4i v[P];
    int next;
    __device__ __forceinline__ v4i get(int p, unsigned shift) const {
        const int after = p + 1 < P ? v[p + 1 < P ? p + 1 : p][0] : next;
        return v4i{static_cast<int>(__builtin_amdgcn_alignbyte(v[p][1], v[p][0], shift)),
                   static_cast<int>(__builtin_amdgcn_alignbyte(v[p][2], v[p][1], shift)),
                   static_cast<int>(__builtin_amdgcn_alignbyte(v[p][3], v[p][2], shift)),
                   static_cast<int>(__builtin_amdgcn_alignbyte(after, v[p][3], shift))};
    }
};
// A row's first dword and how many bytes of it lie before the row.
struct RowStart {
    const int8_t *dword;
    unsigned shift;
    __device__ __forceinline__ explicit RowStart(const int8_t *row)
        : dword(row - (reinterpret_cast<uintptr_t>(row) & 3u)), shift(reinterpret_cast<uintptr_t>(row) & 3u) {}
    RowStart() = default;
    template <bool SHIFT, int P>
    __device__ __forceinline__ ShiftedPieces<P> load(int k) const {  // bytes k .. k + 16 P - 1 of the row, k a multiple of four
        ShiftedPieces<P> r;
#pragma unroll
        for (int p = 0; p < P; ++p) r.v[p] = reinterpret_cast<const Dwords16 *>(dword + k + 16 * p)->v;
        r.next = 0;
        if constexpr (SHIFT) r.next = *reinterpret_cast<const int *>(dword + k + (shift ? 16 * P : 16 * P - 4));
        return r;
    }
};

// Bytes k .. k + 15 of a row that ends at K (16 <= K): zeros from there on.  Its last 16 bytes are read and shifted down,
// without a branch, so that the loads of several pieces are in flight together.
struct TailPiece {
    ShiftedPieces<1> raw;
    unsigned shift;
    int drop;
    __device__ __forceinline__ void load(const RowStart &row, int k, int K) {
        const int at = k < K - 16 ? k : K - 16;
        const RowStart from(row.dword + row.shift + at);
        raw = from.load<true, 1>(0);
        shift = from.shift;
        drop = k - at;
    }
    __device__ __forceinline__ v4i get() const {
        const v4i v = raw.get(0, shift);
        const int d = drop >> 2;  // whole dwords, then bytes
        const int w0 = d == 0 ? v[0] : d == 1 ? v[1] : d == 2 ? v[2] : d == 3 ? v[3] : 0,
                  w1 = d == 0 ? v[1] : d == 1 ? v[2] : d == 2 ? v[3] : 0, w2 = d == 0 ? v[2] : d == 1 ? v[3] : 0,
                  w3 = d == 0 ? v[3] : 0;
        return ShiftedPieces<1>{{v4i{w0, w1, w2, w3}}, 0}.get(0, drop & 3);
    }
};

template <int FM, int FN, int WK>
constexpr int split_rows_lds_bytes() {
    return WK * FM * FN * kWave * int(sizeof(v4i));
}

// SHIFT: rows that are not all dword aligned.
template <int FM, int FN, int WK, int EPI, bool EVEN, bool SHIFT, int P>
__global__ __launch_bounds__(64 * WK) void split_i8_rows_kernel(const int8_t *__restrict__ A, const int8_t *__restrict__ W,
                                                                int M, int N, int K, GemmEpilogue ep) {
    constexpr int BLOCKS = FM * FN, PER_WAVE = (BLOCKS + WK - 1) / WK;
    extern __shared__ __attribute__((aligned(16))) v4i split_part[];  // [WK][BLOCKS][kWave]
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int m0 = static_cast<int>(blockIdx.y) * (16 * FM), n0 = static_cast<int>(blockIdx.x) * (16 * FN);
    const int frow = lane % 16, g = lane / 16;
    RowStart ap[FM], wp[FN];  // rows past the edge are computed and discarded
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int m = m0 + 16 * i + frow;
        ap[i] = RowStart(A + size_t(m < M ? m : M - 1) * K);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int n = n0 + 16 * j + frow;
        wp[j] = RowStart(W + size_t(n < N ? n : N - 1) * K);
    }
    ShiftedPieces<P> fa[FM], fw[FN];
    const int whole = K / (64 * P);  // steps of 64 bytes; what is left is one more, taken by the wave whose turn it is
    auto issue = [&](int s) {  // step wave + WK * s; past the last: nothing is read, zeros
        const int step = wave + WK * s;
        if (step < whole) {
            const int k = (step * 64 + 16 * g) * P;
#pragma unroll
            for (int i = 0; i < FM; ++i) fa[i] = ap[i].template load<SHIFT, P>(k);
#pragma unroll
            for (int j = 0; j < FN; ++j) fw[j] = wp[j].template load<SHIFT, P>(k);
        } else {
#pragma unroll
            for (int i = 0; i < FM; ++i) fa[i] = ShiftedPieces<P>{};
#pragma unroll
            for (int j = 0; j < FN; ++j) fw[j] = ShiftedPieces<P>{};
        }
    };
    issue(0);
    // Block b = (b / FN, b % FN) of the tile is finished by wave b % WK; a lane holds row lane % 16, channels 4 g .. 4 g + 3.
    EpilogueOperands eo[PER_WAVE];
    if constexpr (EPI != EPI_I32) {
#pragma unroll
        for (int p = 0; p < PER_WAVE; ++p) {
            const int b = wave + WK * p;
            if (b < BLOCKS)
                eo[p] = load_epilogue_operands<EPI>(ep, m0 + 16 * (b / FN) + frow, n0 + 16 * (b % FN) + 4 * g, M, N);
        }
    }
    v4i acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    auto multiply = [&](const v4i *a, const v4i *w) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[j], a[i], acc[i][j], 0, 0, 0);
    };
    auto multiply_step = [&]() {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            v4i a[FM], w[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) a[i] = SHIFT ? fa[i].get(p, ap[i].shift) : fa[i].v[p];
#pragma unroll
            for (int j = 0; j < FN; ++j) w[j] = SHIFT ? fw[j].get(p, wp[j].shift) : fw[j].v[p];
            multiply(a, w);
        }
    };
    // what is left of K: P steps of 64 bytes or fewer, dealt to the waves behind the whole steps
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int k0 = whole * 64 * P + 64 * p;
        if (k0 >= K || wave != (whole + p) % WK) continue;
        TailPiece ta[FM], tw[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) ta[i].load(ap[i], k0 + 16 * g, K);
#pragma unroll
        for (int j = 0; j < FN; ++j) tw[j].load(wp[j], k0 + 16 * g, K);
        v4i a[FM], w[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) a[i] = ta[i].get();
#pragma unroll
        for (int j = 0; j < FN; ++j) w[j] = tw[j].get();
        multiply(a, w);
    }
    const int steps = (whole + WK - 1) / WK;
    for (int s = 1; s < steps; ++s) {
        multiply_step();
        issue(s);
    }
    multiply_step();
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) split_part[(wave * BLOCKS + i * FN + j) * kWave + lane] = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PER_WAVE; ++p) {
        const int b = wave + WK * p;
        if (b >= BLOCKS) continue;
        v4i sum = split_part[b * kWave + lane];
#pragma unroll
        for (int w = 1; w < WK; ++w) sum += split_part[(w * BLOCKS + b) * kWave + lane];
        epilogue_store4_loaded<EPI, EVEN>(ep, eo[p], m0 + 16 * (b / FN) + frow, n0 + 16 * (b % FN) + 4 * g, M, N, sum);
    }
}

template <int FM, int FN, int WK, int P, int EPI, bool EVEN>
static int32_t launch_split_rows(hipq_ctx *ctx, const int8_t *a, const int8_t *w, int M, int N, int K, const GemmEpilogue &ep) {
    constexpr int kLds = split_rows_lds_bytes<FM, FN, WK>();
    static_assert(kLds <= 65536, "no more LDS than a kernel may have without asking");
    const bool dwords = K % 4 == 0 && ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w)) & 3u) == 0;
    auto kernel = dwords ? split_i8_rows_kernel<FM, FN, WK, EPI, EVEN, false, P> : split_i8_rows_kernel<FM, FN, WK, EPI, EVEN, true, P>;
    const dim3 grid((N + 16 * FN - 1) / (16 * FN), (M + 16 * FM - 1) / (16 * FM));
    hipLaunchKernelGGL(kernel, grid, dim3(64 * WK), kLds, ctx->stream, a, w, M, N, K, ep);
    return check_launch("gemm_i8 (split)");
}

}  // namespace hipq
