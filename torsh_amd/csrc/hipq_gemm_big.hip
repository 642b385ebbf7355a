// int8 GEMM on fragment-packed operands for products with more tiles than compute units: large tiles staged through LDS.
//
// A workgroup of four waves (WM x WN) owns BM x BN = (32 WM FM) x (32 WN FN) outputs, a wave FM x FN accumulator blocks.
// The packed layout (hipq_gemm_packed.h) makes a fragment - one MFMA operand, 32 rows x 32 bytes of K - one contiguous
// KiB, so a fill is one buffer_load ... lds per fragment (memory to LDS, no registers) and a read is one ds_read_b128 per
// lane at lane * 16: no swizzle, no bank conflict, no address arithmetic.  NS stages of SK k blocks are in LDS; a stage is
// requested NS - 1 stages ahead, by all waves alike, and one barrier per stage publishes it.
//
// Why it beats the forms without LDS here: what a compute unit pulls from its L2 per MFMA falls with the tile (0.375 KiB
// for 128 x 256, against 0.75 KiB for the 128 x 64 tiles whose operands go straight to registers), and that traffic is
// both that path's limit and much of the power the clock is paid with.  Two workgroups share a compute unit (72 KiB of
// LDS, 256 registers a wave), so one converts and stores while the other multiplies.
// Measured, fp32 out, us against the 128 x 64 tiles: 4096 x 11008 x 4096 270 -> 174 (2.1 POP/s), 8192^3 755 -> 450 (2.44),
// 8192 x 3072 x 768 37 -> 31, 2048 x 4096 x 4096 43 -> 38, 256 x 32000 x 4096 49 -> 41.  What bounds it: power.  The matrix
// pipes are busy 71 % of the cycles at 1.62 GHz; 256 x 256 tiles (256 accumulator registers a wave, one wave per SIMD: 58 %
// of the cycles at 1.82 GHz; eight waves of 128 x 64 outputs) deliver the same 2.35-2.5 POP/s at 8192^3, and no more than
// these at 4096 x 11008 x 4096, where their 688 tiles leave the last of three rounds two thirds full.
//
// The order of a k block is fixed: the reads of the next k block's fragments and the fills are spread over its MFMAs, the
// reads in the order of use (at a stage's end behind the barrier, which itself goes behind two MFMAs).  The fills are inline assembly: told of them, the compiler
// would put a wait for all of them in front of every LDS read.
#include "hipq_gemm_kernels.h"

namespace hipq {

// One fragment (1 KiB): memory -> LDS.  rsrc: buffer descriptor; lds: byte address in LDS.
__device__ __forceinline__ void fill_fragment(v4i rsrc, uint32_t lds, int voff, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(rsrc),
                 "s"(soff)
                 : "memory", "m0");
}

template <int WM, int WN, int FM, int FN, int SK, int NS, int EPI, bool EVEN>
__global__ __launch_bounds__(64 * WM * WN, FM * FN > 8 ? 1 : 2) void gemm_i8_packed_lds_kernel(const int8_t *__restrict__ PA,
                                                                                       const int8_t *__restrict__ PW, int M,
                                                                                       int N, int K, int group_m,
                                                                                       GemmEpilogue ep) {
    constexpr int NW = WM * WN;
    constexpr int RA = WM * FM, RW = WN * FN, F = RA + RW;  // fragments per k block
    static_assert(RA % NW == 0 && RW % NW == 0, "fills divide evenly between the waves");
    constexpr int L = SK * F / NW;                          // fills per wave and stage
    constexpr int PART = L / SK;                            // ... and k block
    constexpr int NF = FM + FN, NM = FM * FN;               // reads and MFMAs per wave and k block
    static_assert(NM >= NF && SK >= 2 && SK % 2 == 0 && NS >= 3, "pipeline shape");
    constexpr int STAGE = SK * F * 1024;
    constexpr int LAG = (NS - 3) * L + (SK - 1) * PART;     // fills younger than the next stage's at its barrier
    static_assert(LAG < 64, "vmcnt is a 6-bit counter");
    extern __shared__ __attribute__((aligned(1024))) int8_t lds[];

    const int KB = static_cast<int>(packed_k_blocks(K));
    const int rbA = (M + 31) / 32, rbW = (N + 31) / 32;
    const int tiles_m = (rbA + RA - 1) / RA, tiles_n = (rbW + RW - 1) / RW, ntiles = tiles_m * tiles_n;
    // An XCD (workgroups b, b + 8, ...) takes a contiguous run of the tiles, ordered in bands of group_m row tiles and
    // column by column inside a band, so that the tiles its compute units hold at one time share rows and columns.
    const int per = (ntiles + 7) / 8;
    const int lin = static_cast<int>(blockIdx.x % 8) * per + static_cast<int>(blockIdx.x / 8);
    if (static_cast<int>(blockIdx.x / 8) >= per || lin >= ntiles) return;
    const int band = lin / (group_m * tiles_n), in_band = lin % (group_m * tiles_n);
    const int band_m = tiles_m - band * group_m < group_m ? tiles_m - band * group_m : group_m;
    const int tile_m = band * group_m + in_band % band_m, tile_n = in_band / band_m;
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int wm = wave % WM, wn = wave / WM;
    const int m0 = (tile_m * RA + wm * FM) * 32, n0 = (tile_n * RW + wn * FN) * 32;  // of this wave

    // Fill i of a stage, wave w: fragment (NW i + w) % F of k block (NW i + w) / F: operand and k block depend on i only.
    auto descriptor = [](const int8_t *p, int bytes) {
        const uint64_t a = reinterpret_cast<uint64_t>(p);
        return v4i{__builtin_amdgcn_readfirstlane(static_cast<int>(a)),
                   __builtin_amdgcn_readfirstlane(static_cast<int>(a >> 32) & 0xffff), bytes, 0x00020000};
    };
    const v4i ra = descriptor(PA, rbA * KB * 1024), rw = descriptor(PW, rbW * KB * 1024);
    int src[F / NW];  // first k block of the fragment this wave fills as number NW i + wave
#pragma unroll
    for (int i = 0; i < F / NW; ++i) {
        const int f = NW * i + wave;
        int rb = i < RA / NW ? tile_m * RA + f : tile_n * RW + f - RA;
        const int last = (i < RA / NW ? rbA : rbW) - 1;
        rb = rb < last ? rb : last;  // row blocks past the matrix repeat the last one: computed and discarded
        src[i] = rb * KB * 1024;
    }
    const int voff = lane * 16;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) int8_t *)lds));
    const int nst = KB / SK;
    int fill_stage = 0, fill_buf = 0;  // next stage to request, byte offset of its buffer
    auto fill_one = [&](int j) {       // fill j of stage fill_stage
        const int i = j % (F / NW), kk = j / (F / NW);
        fill_fragment(i < RA / NW ? ra : rw, lds0 + fill_buf + (kk * F + NW * i + wave) * 1024, voff,
                      src[i] + (fill_stage * SK + kk) * 1024);
    };
    auto next_fill_stage = [&]() {
        ++fill_stage;
        fill_buf = fill_buf + STAGE == NS * STAGE ? 0 : fill_buf + STAGE;
    };

    v4i fa[2][FM], fw[2][FN];
    const int8_t *const my_a = lds + wm * FM * 1024 + voff, *const my_w = lds + (RA + wn * FN) * 1024 + voff;
    auto read_one = [&](int set, int q, int at) {  // q-th fragment of the k block at byte `at`: A0, all of W, the rest of A
        if (q == 0 || q > FN) {
            const int i = q == 0 ? 0 : q - FN;
            fa[set][i] = *reinterpret_cast<const v4i *>(my_a + at + i * 1024);
        } else {
            fw[set][q - 1] = *reinterpret_cast<const v4i *>(my_w + at + (q - 1) * 1024);
        }
    };
    v16i acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
        if (s < nst) {
#pragma unroll
            for (int j = 0; j < L; ++j) fill_one(j);
            next_fill_stage();
        }
    if (nst >= NS - 1)
        wait_vmcnt<(NS - 2) * L>();
    else
        wait_vmcnt<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int t = 0; t < NF; ++t) read_one(0, t, 0);

    // Behind which MFMA of a k block the q-th read goes: in the order of use (MFMAs run row block by row block), spread
    // over the block, at a stage's end behind the barrier.
    constexpr int LEAD = 2;  // MFMAs ahead of the barrier
    auto read_slot = [](int q, bool last) {
        if (!last) return q * (NM - 1) / (NF + 1);
        return LEAD - 1 + q * (NM - LEAD) / NF;
    };
    int at = 0;  // byte offset of the stage being multiplied
    for (int s = 0; s < nst; ++s) {
        const bool filling = fill_stage < nst;
        const int next = at + STAGE == NS * STAGE ? 0 : at + STAGE;
#pragma unroll
        for (int kk = 0; kk < SK; ++kk) {
            const int set = kk % 2;
#pragma unroll
            for (int t = 0; t < NM; ++t) {
                const int i = t / FN, j = t % FN;
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[set][i], fw[set][j], acc[i][j], 0, 0, 0);
                if (t + 1 == LEAD && kk == SK - 1) {
                    // The next stage has landed (this wave's share of it; the barrier adds the others'), and this
                    // stage's last fragments are in registers: behind the barrier its buffer may be filled again.
                    if (filling)
                        wait_vmcnt<LAG>();
                    else
                        wait_vmcnt<0>();
                    wait_lgkmcnt0();
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                }
#pragma unroll
                for (int q = 0; q < NF; ++q)
                    if (t == read_slot(q, kk == SK - 1))
                        read_one(set ^ 1, q, kk == SK - 1 ? next : at + (kk + 1) * (F * 1024));
                if (filling) {
#pragma unroll
                    for (int f = 0; f < PART; ++f)
                        if (t == (f * NM + NM / 2) / PART) fill_one(kk * PART + f);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (filling) next_fill_stage();
        at = next;
    }

    // Epilogue.
    float swv[FN], bv[FN], sa0 = 1.0f;
    int nn[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        nn[j] = n0 + j * 32 + lane % 32;
        const int nc = nn[j] < N ? nn[j] : N - 1;
        swv[j] = 1.0f;
        bv[j] = 0.0f;
        if constexpr (EPI != EPI_I32) {
            swv[j] = ep.sw[nc];
            if (ep.bias) bv[j] = ep.bias[nc];
        }
    }
    if constexpr (EPI != EPI_I32)
        if (!ep.sa_per_row) sa0 = ep.sa ? ep.sa[0] : ep.sa_scalar;
    bool interior = false;
    if constexpr (EPI != EPI_I8) interior = m0 + FM * 32 <= M && n0 + FN * 32 <= N && ep.residual == nullptr;
    if (interior) {
        if constexpr (EPI != EPI_I8) {
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                v16i own[1][FN];
#pragma unroll
                for (int j = 0; j < FN; ++j) own[0][j] = acc[i][j];
                store_block_interior<FN, EPI>(own, ep, N, m0 + i * 32, n0, lane, swv, bv, sa0);
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            v16i own[1][FN];
#pragma unroll
            for (int j = 0; j < FN; ++j) own[0][j] = acc[i][j];
            store_tile<1, FN, 1, EPI, EVEN>(own, ep, M, N, m0 + i * 32, 0, lane, nn, swv, bv, sa0);
        }
    }
}

template <int WM, int WN, int FM, int FN, int SK, int NS, int EPI, bool EVEN>
static int32_t launch_packed_lds(hipq_ctx *ctx, const int8_t *pa, const int8_t *pw, int M, int N, int K,
                                 const GemmEpilogue &ep) {
    constexpr int RA = WM * FM, RW = WN * FN, kLds = NS * SK * (RA + RW) * 1024;
    auto kernel = gemm_i8_packed_lds_kernel<WM, WN, FM, FN, SK, NS, EPI, EVEN>;
    static bool configured[16] = {false};  // per device: raise the dynamic LDS limit once
    if (ctx->device < 16 && !configured[ctx->device]) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
        if (e != hipSuccess)
            return fail(HIPQ_DEVICE_ERROR, "gemm_i8 (packed, LDS): cannot reserve %d bytes of LDS: %s", kLds,
                        hipGetErrorString(e));
        configured[ctx->device] = true;
    }
    const int tiles_m = ((M + 31) / 32 + RA - 1) / RA, tiles_n = ((N + 31) / 32 + RW - 1) / RW;
    const int group_m = tiles_m < 8 ? tiles_m : 8;
    hipLaunchKernelGGL(kernel, dim3((tiles_m * tiles_n + 7) / 8 * 8), dim3(64 * WM * WN), kLds, ctx->stream, pa, pw, M, N, K, group_m,
                       ep);
    return check_launch("gemm_i8 (packed, LDS)");
}

template <int EPI, bool EVEN>
static int32_t launch_form(hipq_ctx *ctx, bool tall, const int8_t *pa, const int8_t *pw, int M, int N, int K,
                           const GemmEpilogue &ep) {
    if (tall) return launch_packed_lds<2, 2, 4, 2, 2, 3, EPI, EVEN>(ctx, pa, pw, M, N, K, ep);
    return launch_packed_lds<2, 2, 2, 4, 2, 3, EPI, EVEN>(ctx, pa, pw, M, N, K, ep);
}

int32_t gemm_packed_lds(hipq_ctx *ctx, bool tall, const int8_t *pa, const int8_t *pw, int M, int N, int K,
                        const GemmEpilogue &ep, int epi, bool even) {
    if (epi == EPI_I32) return launch_form<EPI_I32, false>(ctx, tall, pa, pw, M, N, K, ep);
    if (epi == EPI_F32) return launch_form<EPI_F32, false>(ctx, tall, pa, pw, M, N, K, ep);
    if (even) return launch_form<EPI_I8, true>(ctx, tall, pa, pw, M, N, K, ep);
    return launch_form<EPI_I8, false>(ctx, tall, pa, pw, M, N, K, ep);
}

}  // namespace hipq
