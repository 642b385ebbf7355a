// The prepared transformer stack on few tokens, all layers in one launch: eight teams, the workgroups of one XCD each, take an
// eighth of the rows through every layer.
//
// As separate launches a layer of few tokens is five kernels of 4 to 7 us, each a launch, a cold start on weights that nobody
// has asked for yet, and a trip through memory to the next one's compute units on the other XCDs.  Rows do not meet in this
// stack, so nothing has to leave an XCD: a team's 32 workgroups split the columns of every product, hand their results on through
// the L2 they share and meet there (a flag per workgroup, one line per team, read past the L1).  While it waits, a workgroup's
// share of the next product's weights is already on its way into registers.  The price is that every XCD streams all
// the weights; they come from the memory-side cache for all but the first.
//
// Per layer: LayerNorm + quantize + qkv | quantize V + out-projection + skip | LayerNorm + quantize + fc1 + GELU and row maxima |
// GELU codes | fc2 + skip.  The row operations in front of a product are repeated by every workgroup, a row per wave, as in
// row_op_split_kernel, whose arithmetic and orders these are: the bits of the separate kernels.
//
// A team needs all its workgroups on the device at once, which other work may prevent (another stream's team is enough).
// So it first counts itself: either the last workgroup to arrive finds that nobody has stopped waiting, and all 32 go on and
// wait for nothing but each other from there on; or somebody stops waiting first, all of them leave without having touched
// anything, and the kernel behind this one takes the team's rows through the layers with those of its workgroups that are there.
#include "hipq_gemm_kernels.h"
#include "hipq_internal.h"
#include "hipq_panel_norm.h"
#include "hipq_quantize_rows.h"
#include "hipq_team_words.h"

namespace hipq {
namespace {

constexpr int kTeams = static_cast<int>(kCtxTeams);
constexpr int kTeamSize = 32;     // workgroups of a team
constexpr int kTeamWaves = 16;    // waves of a workgroup: the first multiply, the others take the rows
constexpr int kTeamProducts = 6;  // waves that multiply
constexpr int kTeamRowWaves = kTeamWaves - kTeamProducts;
constexpr int kTeamRows = 16;     // rows of a team at most
static_assert(kTeamTokens == size_t(kTeams) * kTeamRows, "tokens of all teams");
constexpr int kTeamLayers = 24;   // layers of one launch (their pointers are kernel arguments)
constexpr int kTeamFloats = 3;    // float4 a lane per row: d_model <= 768
constexpr int kTeamColumns = 3;   // column blocks of 32 a workgroup: N <= 3072
constexpr int kTeamSteps = 8;     // pairs of k blocks a wave: K <= 3072
constexpr int kTeamRowSteps = 2;  // the same where K is d_model
static_assert(kTeamLayers * 5 < int(kTeamPhases), "five meetings a layer");
constexpr int kPastL1 = /*sc1*/ 16;

// Looks at the verdict before a workgroup stops waiting for its team, some 0.1 us each.  Beside ordinary kernels, whose workgroups make
// room one after the other, a team assembles within that and then has its compute units: 77 tokens, d 768, us by 64 / 512 / 4096 looks
// beside bf16 products of 4096^3 603 / 604 / 603 (separate kernels 5400: each waits again), an addition over 512 MB 922 / 448 / 447
// (1170), Linears of 4096 x 11008 x 4096 602 / 401 / 401 (2450).  Where a workgroup that holds 128 KB of LDS for milliseconds sits on
// every XCD, waiting is in vain: 1 / 256 / 1024 / 4096 looks 460 / 490 / 572 / 900 (separate kernels 345 to 365).
constexpr int kAssemblyLimit = 512;

struct StackTeam {
    hipq_block_weights blocks[kTeamLayers];
    float *x, *qkv, *maxima;
    int8_t *codes;
    uint32_t *words, *wait_error;
    int layers, qkv_done, tokens, rows, d, d_ff, spin_limit, assembly_limit, gather_looks;
    float eps;
};
static_assert(sizeof(StackTeam) <= 4096, "kernel arguments");

__device__ __forceinline__ __amdgpu_buffer_rsrc_t team_buffer(const void *base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00020000);
}

// Words of a team: how many workgroups have ever arrived (32 a launch), what was decided about the last launch - its number and
// whether the team goes on - and, where it does not, who has come to the kernel behind this one.
constexpr int kTeamArrivals = 0, kTeamVerdict = 1, kTeamGather = 2, kTeamGo = 1, kTeamApart = 2;

// One lane of a workgroup: arrives and waits for the verdict on this launch, whose number is left in `launch`.
__device__ __forceinline__ bool team_assembles(uint32_t *words, int spin_limit, uint32_t *launch) {
    const uint32_t before = __hip_atomic_fetch_add(words + kTeamArrivals, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t n = before / kTeamSize;
    *launch = n;
    if (before % kTeamSize == 0) __hip_atomic_store(words + kTeamGather, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint32_t *verdict = words + kTeamVerdict, seen = 0;
    auto decided = [&] { return seen != 0 && (seen >> 2) == n; };
    auto decide = [&](uint32_t v) {  // unless it has been decided already
        seen = __hip_atomic_load(verdict, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        while (!decided())
            if (__hip_atomic_compare_exchange_strong(verdict, &seen, n << 2 | v, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT))
                seen = n << 2 | v;
    };
    if (before % kTeamSize == kTeamSize - 1) {
        decide(kTeamGo);
    } else {
        for (int spin = 0; spin < spin_limit && !decided(); ++spin) {
            __builtin_amdgcn_s_sleep(1);
            seen = __hip_atomic_load(verdict, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (!decided()) decide(kTeamApart);
    }
    return (seen & 3u) == kTeamGo;
}

__device__ __forceinline__ uint32_t team_xcc_id() {
    uint32_t v;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(v));
    return v;
}

// Maximum over a row of 16 lanes, in every lane.
__device__ __forceinline__ float lane_row_max(float v) {
    v = fmaxf(v, lane_move<0xB1>(v));   // quad_perm [1, 0, 3, 2]
    v = fmaxf(v, lane_move<0x4E>(v));   // quad_perm [2, 3, 0, 1]
    v = fmaxf(v, lane_move<0x141>(v));  // row_half_mirror
    return fmaxf(v, lane_move<0x140>(v));  // row_mirror
}

// Waves have roles, because a wave's loads return in the order of their requests: the six that multiply ask for the next
// product's weights as soon as they have parked their partial sums (and touch those of the one after it, so that they are in the
// L2 by then), the ten others poll, run the row operations, and finish and store results, and never wait for a weight.
template <bool EVEN>
__global__ __launch_bounds__(1024) void stack_team_kernel(StackTeam p) {
    constexpr int RC = kTeamFloats, kPiece = kTeamRows + 1;  // (a piece of padding: the lanes of a store hit all banks)
    __shared__ __attribute__((aligned(16))) v4i codes[kTeamColumns * kTeamSize * 2 * kPiece];  // [k block][half][row]
    __shared__ __attribute__((aligned(16))) v4i part[kTeamProducts][2 * kTeamColumns][kWave];
    __shared__ __attribute__((aligned(16))) float4 gain[RC * 64], offset[RC * 64];  // of the LayerNorm ahead
    __shared__ float col_scale[2][kTeamColumns * 32], col_bias[2][kTeamColumns * 32];  // of this product and the next
    __shared__ float row_scale[kTeamRows], row_inv[kTeamRows];
    __shared__ int together;
    int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const bool multiplies = wave < kTeamProducts;
    const int rw = wave - kTeamProducts;  // of the waves that take rows
    const int team = static_cast<int>(blockIdx.x) % kTeams, me = static_cast<int>(blockIdx.x) / kTeams;
    const int T = p.rows, row0 = team * T;
    if (row0 >= p.tokens) return;
    const int R = T < p.tokens - row0 ? T : p.tokens - row0;
    const int d = p.d, dblocks = d / 32, fblocks = p.d_ff / 32;
    uint32_t *words = p.words + team * kCtxTeamWords;
    const __amdgpu_buffer_rsrc_t rflags = team_buffer(words + kCtxTeamFlags, kTeamSize * 4);
    const __amdgpu_buffer_rsrc_t rx = team_buffer(p.x + size_t(row0) * d, R * d * 4);
    const __amdgpu_buffer_rsrc_t rqkv = team_buffer(p.qkv + size_t(row0) * 3 * d, R * 3 * d * 4);
    const __amdgpu_buffer_rsrc_t rmaxima = team_buffer(p.maxima + size_t(team) * T * fblocks * 2, T * fblocks * 8);  // [16 columns][row]
    const __amdgpu_buffer_rsrc_t rcodes = team_buffer(p.codes + size_t(team) * T * p.d_ff, T * p.d_ff);  // [k block][half][row][16]

    // A product is v_mfma_i32_16x16x64_i8, as the rows are 16 at most.  Operands: a lane's 16 bytes are of row or column lane % 16
    // and of quarter lane / 16 of two consecutive k blocks.  Results: column lane % 16, rows `mine` + 0 .. 3.
    int mine = 4 * (lane / 16), fragment = lane / 16 * 512 + lane % 16 * 16;
    // Columns: this workgroup has blocks me, me + 32, ... of a product's 32-column blocks.
    auto column_block = [&](int j) { return me + kTeamSize * j; };
    const std::integral_constant<int, 1> narrow;
    const std::integral_constant<int, kTeamColumns> wide;
    const std::integral_constant<int, kTeamRowSteps> shallow;
    const std::integral_constant<int, kTeamSteps> deep;


    if (multiplies) {
        v4i fw[2 * kTeamSteps];
        uint32_t touched[kTeamColumns] = {0, 0, 0};
#pragma unroll
        for (int i = 0; i < 2 * kTeamSteps; ++i) fw[i] = v4i{0, 0, 0, 0};
        // This wave's fragments of a product's weights.
        auto request = [&](auto steps, auto columns, const int8_t *w, int nblocks, int kblocks) {
            constexpr int STEPS = decltype(steps)::value, CB = decltype(columns)::value;
            static_assert(STEPS * CB <= kTeamSteps, "registers for the fragments");
            const __amdgpu_buffer_rsrc_t rw_ = team_buffer(w, nblocks * kblocks * 1024);
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const int kb = 2 * (wave + kTeamProducts * s);
#pragma unroll
                for (int jc = 0; jc < 2 * CB; ++jc)
                    if (kb < kblocks && column_block(jc / 2) < nblocks)  // (the others are not multiplied or not looked at)
                        fw[s * 2 * CB + jc] = __builtin_bit_cast(
                            v4i, __builtin_amdgcn_raw_buffer_load_b128(rw_, fragment, (column_block(jc / 2) * kblocks + kb) * 1024 + jc % 2 * 256, 0));
            }
        };
        // One dword of every line of the workgroup's share of a product's weights.
        auto touch = [&](auto columns, const int8_t *w, int nblocks, int kblocks) {
            constexpr int CB = decltype(columns)::value;
            const __amdgpu_buffer_rsrc_t rw_ = team_buffer(w, nblocks * kblocks * 1024);
#pragma unroll
            for (int u = 0; u < kTeamColumns; ++u) {
                const int line = CB == 1 ? wave * kWave + lane + u * (kTeamProducts * kWave) : wave * kWave + lane;
                const int j = CB == 1 ? 0 : u;
                if (line < kblocks * 8 && column_block(j) < nblocks)
                    touched[u] = __builtin_amdgcn_raw_buffer_load_b32(rw_, line * 128, column_block(j) * kblocks * 1024, 0);
            }
        };
        auto settle = [&] {
#pragma unroll
            for (int u = 0; u < kTeamColumns; ++u) {
                const uint32_t t = touched[u];
                asm volatile("" ::"v"(t));
            }
        };
        // Multiplies this wave's k blocks and parks the partial blocks.  (Rows past the team's hold whatever is there; their results
        // are not looked at.)
        auto multiply = [&](auto steps, auto columns, int nblocks, int kblocks, auto touch_next) {
            constexpr int STEPS = decltype(steps)::value, CB = decltype(columns)::value;
            __syncthreads();  // the rows are there
            touch_next();
            __syncthreads();  // and their codes
            v4i acc[2 * CB];
#pragma unroll
            for (int jc = 0; jc < 2 * CB; ++jc) acc[jc] = v4i{0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const int kb = 2 * (wave + kTeamProducts * s);
                if (kb >= kblocks) break;
                const v4i fa = codes[(kb * 2 + lane / 16) * kPiece + lane % kTeamRows];
#pragma unroll
                for (int jc = 0; jc < 2 * CB; ++jc)
                    acc[jc] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa, fw[s * 2 * CB + jc], acc[jc], 0, 0, 0);
            }
#pragma unroll
            for (int jc = 0; jc < 2 * CB; ++jc)
                if (column_block(jc / 2) < nblocks) part[wave][jc][lane] = acc[jc];
            __syncthreads();
            settle();
        };
        auto others = [&](int barriers) {  // the row waves' further ones of a phase
            for (int i = 0; i < barriers; ++i) __syncthreads();
            // (addresses are made again in every phase: kept from layer to layer, they would take more registers than there are)
            asm volatile("" : "+v"(lane), "+v"(fragment)::"memory");
        };
        if (p.qkv_done)
            request(shallow, narrow, p.blocks[0].w_out, dblocks, dblocks);
        else
            request(shallow, wide, p.blocks[0].w_qkv, 3 * dblocks, dblocks);
        __syncthreads();
        if (!together) return;
#pragma unroll 1
        for (int l = 0; l < p.layers; ++l) {
            const hipq_block_weights &b = p.blocks[l];
            const bool last = l + 1 == p.layers;
            if (l > 0 || !p.qkv_done) {
                multiply(shallow, wide, 3 * dblocks, dblocks, [&] { touch(narrow, b.w_out, dblocks, dblocks); });
                request(shallow, narrow, b.w_out, dblocks, dblocks);
                others(2);
            }
            multiply(shallow, narrow, dblocks, dblocks, [&] { touch(wide, b.w_fc1, fblocks, dblocks); });
            request(shallow, wide, b.w_fc1, fblocks, dblocks);
            others(2);
            multiply(shallow, wide, fblocks, dblocks, [&] { touch(narrow, b.w_fc2, dblocks, fblocks); });
            request(deep, narrow, b.w_fc2, dblocks, fblocks);
            others(5);  // (the scales of GELU's rows, and another meeting)
            multiply(deep, narrow, dblocks, fblocks, [&] {
                if (!last) touch(wide, p.blocks[l + 1].w_qkv, 3 * dblocks, dblocks);
            });
            if (last) break;
            request(shallow, wide, p.blocks[l + 1].w_qkv, 3 * dblocks, dblocks);
            others(2);
        }
        return;
    }

    // Phases are numbered through the launches of the team; the low four bits of a flag name the XCD.
    const uint32_t xcc = team_xcc_id();
    uint32_t phase = 0;
    if (wave == kTeamWaves - 1) {
        uint32_t launch = 0;
        const bool go = lane == 0 && team_assembles(words, p.assembly_limit, &launch);
        if (lane == 0) together = go;
        phase = team_flag(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(launch))), 0);
    }
    bool lost = false;  // (of the wave that polls)
    auto acknowledged = [] {  // this wave's stores have reached the L2
        asm volatile("" ::: "memory");
        wait_vmcnt<0>();
        asm volatile("" ::: "memory");
    };
    auto meet = [&] {
        phase += team_flag(0, 1);
        __syncthreads();
        if (wave == kTeamWaves - 1 && !lost) {
            if (lane == 0) __builtin_amdgcn_raw_buffer_store_b32(static_cast<int>(phase | xcc), rflags, me * 4, 0, 0);
            bool all = false;
            uint32_t seen = 0;
            for (int spin = 0; spin <= p.spin_limit && !all; ++spin) {
                asm volatile("" ::: "memory");
                seen = static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b32(rflags, lane % kTeamSize * 4, 0, kPastL1));
                all = __all(team_flag_reached(seen, phase));
            }
            lost = !all || !__all((seen & 15u) == xcc);
        }
        __syncthreads();
        // (addresses are made again in every phase: kept from layer to layer, they would take more registers than there are)
        asm volatile("" : "+v"(lane), "+v"(mine), "+v"(fragment)::"memory");
    };

    // Scales and biases of a product's columns and, for a LayerNorm in front of it, its vectors: three of the waves that take rows
    // ask for them while the product before it runs, and leave them in LDS behind it.
    const bool fetches = rw >= 6 && rw < 9;
    AnyFloat4 next_gain, next_offset;
    float next_scale = 0.0f, next_bias = 0.0f;
    int product = 0;  // parity of the product whose scales are in use
    auto ask_vectors = [&](const float *scales, const float *biases, int nblocks, bool norm, const float *gamma, const float *beta) {
        if (!fetches) return;
        const int at = (rw - 6) * kWave + lane, block = column_block(at / 32);
        if (at < kTeamColumns * 32 && block < nblocks) {
            next_scale = scales[block * 32 + at % 32];
            next_bias = biases ? biases[block * 32 + at % 32] : 0.0f;
        }
        if (norm && at < d / 4) {  // (y * 1.0f and y + -0.0f are y, bit for bit)
            next_gain = gamma ? reinterpret_cast<const AnyFloat4 *>(gamma)[at] : AnyFloat4{1.0f, 1.0f, 1.0f, 1.0f};
            next_offset = beta ? reinterpret_cast<const AnyFloat4 *>(beta)[at] : AnyFloat4{-0.0f, -0.0f, -0.0f, -0.0f};
        }
    };
    auto leave_vectors = [&](bool norm) {
        product ^= 1;
        if (!fetches) return;
        const int at = (rw - 6) * kWave + lane;
        if (at < kTeamColumns * 32) {
            col_scale[product][at] = next_scale;
            col_bias[product][at] = next_bias;
        }
        if (norm && at < d / 4) {
            gain[at] = make_float4(next_gain.x, next_gain.y, next_gain.z, next_gain.w);
            offset[at] = make_float4(next_offset.x, next_offset.y, next_offset.z, next_offset.w);
        }
    };
    // The codes of the team's rows into LDS, in fragment order, a row per wave.
    auto row_codes = [&](auto norm, const __amdgpu_buffer_rsrc_t &rows, int ld, int first) {
        constexpr int kRounds = (kTeamRows + kTeamRowWaves - 1) / kTeamRowWaves;
        const PanelColumns<RC, false> c(lane, dblocks);
        v4i raw[kRounds][RC];
#pragma unroll
        for (int u = 0; u < kRounds; ++u) {
            const int row = rw + u * kTeamRowWaves;
            if (row < R) {
#pragma unroll
                for (int i = 0; i < RC; ++i)
                    raw[u][i] = __builtin_bit_cast(
                        v4i, __builtin_amdgcn_raw_buffer_load_b128(rows, c.real[i] ? c.at(i) * 4 : 0x7fffffff,
                                                                   (row * ld + first) * 4, kPastL1));
            }
        }
        acknowledged();
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kRounds; ++u) {
            const int row = rw + u * kTeamRowWaves;
            if (row >= R) break;
            float4 v[RC];
#pragma unroll
            for (int i = 0; i < RC; ++i) {  // (a bit cast of a vector's element takes its first one)
                const int t0 = raw[u][i][0], t1 = raw[u][i][1], t2 = raw[u][i][2], t3 = raw[u][i][3];
                v[i] = make_float4(__builtin_bit_cast(float, t0), __builtin_bit_cast(float, t1), __builtin_bit_cast(float, t2),
                                   __builtin_bit_cast(float, t3));
            }
            uint32_t q[RC];
            float scale;
            if constexpr (decltype(norm)::value) {
                PanelAffine<RC> affine;
#pragma unroll
                for (int i = 0; i < RC; ++i)
                    if (c.real[i]) {
                        affine.g[i] = gain[c.at(i) / 4];
                        affine.b[i] = offset[c.at(i) / 4];
                    }
                scale = panel_norm_quantize<EVEN>(v, c, affine, p.eps, q);
            } else {
                scale = row_range_quantize<EVEN>(v, c, q);
            }
            if (lane == 0) row_scale[row] = scale;
            uint32_t *dword = reinterpret_cast<uint32_t *>(codes);
#pragma unroll
            for (int i = 0; i < RC; ++i)
                if (c.real[i]) dword[((c.block[i] * 2 + c.part / 4) * kPiece + row) * 4 + c.part % 4] = q[i];
        }
        __syncthreads();
    };
    // Row wave 2 j + c finishes column half c of block j: its four results of every lane.
    auto finishes = [&](int nblocks) { return rw >= 0 && rw < 2 * kTeamColumns && column_block(rw / 2) < nblocks; };
    constexpr int kPieces = (kTeamColumns * kTeamSize * 2 * kTeamRows + kTeamRowWaves * kWave - 1) / (kTeamRowWaves * kWave);
    auto column = [&] { return column_block(rw / 2) * 32 + rw % 2 * 16 + lane % 16; };
    auto results = [&](float(&o)[4]) {
        v4i sum = part[0][rw][lane];
#pragma unroll
        for (int w = 1; w < kTeamProducts; ++w) sum += part[w][rw][lane];
        const float sw = col_scale[product][rw * 16 + lane % 16], bias = col_bias[product][rw * 16 + lane % 16];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[i] = static_cast<float>(sum[i]) * (row_scale[mine + i] * sw);
            o[i] = o[i] + bias;
        }
    };
    // Result i of this lane, if its row is one of the team's.
    auto store = [&](float v, const __amdgpu_buffer_rsrc_t &to, int at, int i) {
        if (mine + i < R) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), to, at * 4, 0, 0);
    };
    // The stream's values that this lane finishes: the same in out-projection and fc2, so they stay in registers.
    const bool stream = rw < 2 && finishes(dblocks);
    float res[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (stream) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (mine + i < R)
                res[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, ((mine + i) * d + column()) * 4, 0, 0));
    }
    auto add_to_stream = [&] {
        if (!stream) return;
        float o[4];
        results(o);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            res[i] = o[i] + res[i];
            store(res[i], rx, (mine + i) * d + column(), i);
        }
        acknowledged();
    };
    auto ask_qkv = [&](const hipq_block_weights &b) { ask_vectors(b.s_qkv, b.b_qkv, 3 * dblocks, true, b.ln1_gamma, b.ln1_beta); };
    auto ask_out = [&](const hipq_block_weights &b) { ask_vectors(b.s_out, b.b_out, dblocks, false, nullptr, nullptr); };
    if (p.qkv_done)
        ask_out(p.blocks[0]);
    else
        ask_qkv(p.blocks[0]);
    leave_vectors(!p.qkv_done);
    __syncthreads();
    if (!together) return;
#pragma unroll 1
    for (int l = 0; l < p.layers; ++l) {
        const hipq_block_weights &b = p.blocks[l];
        if (l > 0 || !p.qkv_done) {
            row_codes(std::true_type{}, rx, d, 0);
            ask_out(b);
            __syncthreads();
            if (finishes(3 * dblocks)) {
                float o[4];
                results(o);
#pragma unroll
                for (int i = 0; i < 4; ++i) store(o[i], rqkv, (mine + i) * (3 * d) + column(), i);
                acknowledged();
            }
            leave_vectors(false);
            meet();
        }
        // Stand-in for the attention mixing, which is outside this path: the value slice passes through.
        row_codes(std::false_type{}, rqkv, 3 * d, 2 * d);
        ask_vectors(b.s_fc1, b.b_fc1, fblocks, true, b.ln2_gamma, b.ln2_beta);
        __syncthreads();
        add_to_stream();
        leave_vectors(true);
        meet();
        row_codes(std::true_type{}, rx, d, 0);
        ask_vectors(b.s_fc2, b.b_fc2, dblocks, false, nullptr, nullptr);
        __syncthreads();
        const bool hidden = finishes(fblocks);
        const int hblock = column_block(rw / 2) * 2 + rw % 2;  // of 16 columns
        float h[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (hidden) {
            results(h);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                h[i] = gelu_tanh(h[i]);
                const float m = lane_row_max(fmaxf(fabsf(h[i]), 0.0f));  // (a NaN is no maximum)
                if (lane % 16 == 0) store(m, rmaxima, hblock * T + mine + i, i);
            }
            acknowledged();
        }
        leave_vectors(false);
        meet();
        {
#pragma unroll 1
            for (int row = rw; row < R; row += kTeamRowWaves) {
                float am = 0.0f;
#pragma unroll
                for (int i = 0; i < (2 * kTeamColumns * kTeamSize + kWave - 1) / kWave; ++i) {  // (past the last block: zeros)
                    const int at = lane + kWave * i;
                    am = fmaxf(am, __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                                 rmaxima, at < 2 * fblocks ? (at * T + row) * 4 : 0x7fffffff, 0, kPastL1)));
                }
                am = wave_max(am);
                const float scale = am < FLT_EPSILON ? 1.0f : am / 127.0f;
                if (lane == 0) {
                    row_scale[row] = am <= FLT_MAX ? scale : NAN;
                    row_inv[row] = recip_for_div(scale);
                }
            }
        }
        __syncthreads();
        if (hidden) {
            int q[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float scale = row_scale[mine + i];
                q[i] = scale == scale ? quantize_int_sym<EVEN>(h[i], scale, row_inv[mine + i]) : 0;
            }
            const int qd = lane % 4;
            const uint32_t word = quad_byte_transpose(pack4(q[0], q[1], q[2], q[3]), (qd & 1) ? 0x03070105u : 0x06020400u,
                                                      (qd & 2) ? 0x03020706u : 0x05040100u);
            if (mine + qd < R)
                __builtin_amdgcn_raw_buffer_store_b32(static_cast<int>(word), rcodes,
                                                      (hblock * T + mine + qd) * 16 + lane % 16 / 4 * 4, 0, 0);
            acknowledged();
        }
        meet();
        const bool last = l + 1 == p.layers;
        {
            v4i piece[kPieces];
#pragma unroll
            for (int u = 0; u < kPieces; ++u)
                piece[u] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                                       rcodes, ((u * kTeamRowWaves + rw) * kWave + lane) * 16, 0, kPastL1));
            acknowledged();
            __syncthreads();
            const unsigned by_rows = (65536u + T - 1) / T;  // (i / T for i < 3072 and T <= 16: off by less than 1 / T)
#pragma unroll
            for (int u = 0; u < kPieces; ++u) {
                const unsigned i = (u * kTeamRowWaves + rw) * kWave + lane, at = i * by_rows >> 16;
                if (i < unsigned(fblocks * 2 * T)) codes[at * kPiece + (i - at * T)] = piece[u];
            }
        }
        __syncthreads();
        if (!last) ask_qkv(p.blocks[l + 1]);
        __syncthreads();  // the partial blocks are there
        add_to_stream();
        if (!last) {
            leave_vectors(true);
            meet();
        }
    }
    if (wave == kTeamWaves - 1 && lane == 0 && lost)
        __hip_atomic_store(p.wait_error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The same layers of a team's rows by the workgroups that are there, where the team did not assemble: half the registers and a
// third of the LDS of a compute unit each, so they fit beside other work, and however many have arrived after a few looks, one at
// least, share the columns, 16 at a time per wave; who comes later leaves.  So again they wait for nobody but each other.  GELU's
// results are handed on in fp32, in the rows of qkv, which are used up by then, and the codes' room (3 d + d_ff / 4 >= d_ff floats), and
// every workgroup makes the codes of all rows.  77 tokens, d 768, 12 layers: 426 us with all members, 1046 with one or two (one
// workgroup of 16 waves that ran fc1 twice took 2120).
constexpr int kPresentWaves = 8;
constexpr int kPresentChunk = 12;  // pairs of k blocks in flight
constexpr int kGatherLooks = 256;  // some 15 us
constexpr uint32_t kGatherClosed = 0x80;

// One lane: joins, and waits until it is settled who takes part.  The first to come settles it, and until then the flags are its own.
__device__ __forceinline__ bool present_join(uint32_t *words, uint32_t launch, int looks, int spin_limit, int *rank, int *members) {
    uint32_t *gather = words + kTeamGather;
    uint32_t seen = __hip_atomic_load(gather, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    do {
        if (seen & kGatherClosed) return false;
    } while (!__hip_atomic_compare_exchange_strong(gather, &seen, seen + 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    *rank = static_cast<int>(seen++);
    if (*rank == 0) {
        for (int i = 0; i < kTeamSize; ++i) words[kCtxTeamFlags + i] = team_flag(launch, 0);  // (the team has left them as they were)
        for (int look = 0; look < looks && seen < uint32_t(kTeamSize); ++look) {
            __builtin_amdgcn_s_sleep(1);
            seen = __hip_atomic_load(gather, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("" ::: "memory");
        wait_vmcnt<0>();  // the flags have reached the L2
        asm volatile("" ::: "memory");
        seen = __hip_atomic_fetch_or(gather, kGatherClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) | kGatherClosed;
    }
    for (int spin = 0; spin <= spin_limit && !(seen & kGatherClosed); ++spin) {
        __builtin_amdgcn_s_sleep(1);
        seen = __hip_atomic_load(gather, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    *members = static_cast<int>(seen & ~kGatherClosed);
    return (seen & kGatherClosed) != 0;
}

template <bool EVEN>
__global__ __launch_bounds__(kPresentWaves *kWave, 2) void stack_present_kernel(StackTeam p) {
    constexpr int RC = kTeamFloats, kPiece = kTeamRows + 1, HC = kTeamColumns * kTeamSize * 32 / 256;  // (HC: float4 a lane of d_ff)
    __shared__ __attribute__((aligned(16))) v4i codes[kTeamColumns * kTeamSize * 2 * kPiece];
    __shared__ float row_scale[kTeamRows];
    __shared__ int joined, my_rank, all_members;
    const int team = static_cast<int>(blockIdx.x) % kTeams, T = p.rows, row0 = team * T;
    if (row0 >= p.tokens) return;
    uint32_t *words = p.words + team * kCtxTeamWords;
    const uint32_t verdict = words[kTeamVerdict], launch = verdict >> 2;
    if ((verdict & 3u) != kTeamApart) return;
    if (threadIdx.x == 0) {
        int rank = 0, members = 0;
        joined = present_join(words, launch, p.gather_looks, p.spin_limit, &rank, &members);
        my_rank = rank;
        all_members = members;
    }
    __syncthreads();
    if (!joined) return;
    int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int rank = __builtin_amdgcn_readfirstlane(my_rank), members = __builtin_amdgcn_readfirstlane(all_members);
    const int R = T < p.tokens - row0 ? T : p.tokens - row0;
    const int d = p.d, d_ff = p.d_ff, dblocks = d / 32, fblocks = d_ff / 32, mine = 4 * (lane / 16);
    const int beside = d_ff > 3 * d ? d_ff - 3 * d : 0;  // of GELU's results of a row, those that lie where the codes would
    const __amdgpu_buffer_rsrc_t rflags = team_buffer(words + kCtxTeamFlags, kTeamSize * 4);
    const __amdgpu_buffer_rsrc_t rx = team_buffer(p.x + size_t(row0) * d, R * d * 4);
    const __amdgpu_buffer_rsrc_t rqkv = team_buffer(p.qkv + size_t(row0) * 3 * d, R * 3 * d * 4);
    const __amdgpu_buffer_rsrc_t rbeside = team_buffer(p.codes + size_t(team) * T * d_ff, R * beside * 4);
    constexpr int kNowhere = 0x7fffffff;

    uint32_t phase = team_flag(launch, 0);
    const uint32_t xcc = team_xcc_id();
    bool lost = false;  // (of wave 0)
    auto acknowledged = [] {
        asm volatile("" ::: "memory");
        wait_vmcnt<0>();
        asm volatile("" ::: "memory");
    };
    auto meet = [&] {  // behind `acknowledged` of every wave
        phase += team_flag(0, 1);
        __syncthreads();
        if (wave == 0 && !lost) {
            if (lane == 0) __builtin_amdgcn_raw_buffer_store_b32(static_cast<int>(phase | xcc), rflags, rank * 4, 0, 0);
            bool all = false;
            uint32_t seen = 0;
            const bool looks = lane < members;
            for (int spin = 0; spin <= p.spin_limit && !all; ++spin) {
                asm volatile("" ::: "memory");
                seen = static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b32(rflags, lane % kTeamSize * 4, 0, kPastL1));
                all = __all(!looks || team_flag_reached(seen, phase));
            }
            lost = !all || !__all(!looks || (seen & 15u) == xcc);
        }
        __syncthreads();
        asm volatile("" : "+v"(lane)::"memory");
    };
    // The codes of the team's rows into LDS, a row per wave.
    auto row_codes = [&](auto norm, const __amdgpu_buffer_rsrc_t &rows, int ld, int first, const float *gamma, const float *beta) {
        constexpr int kRounds = kTeamRows / kPresentWaves;
        const PanelColumns<RC, false> c(lane, dblocks);
        float4 v[kRounds][RC];
#pragma unroll
        for (int u = 0; u < kRounds; ++u) {
            const int row = wave + u * kPresentWaves;
            if (row < R) {
#pragma unroll
                for (int i = 0; i < RC; ++i)
                    v[u][i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                                             rows, c.real[i] ? c.at(i) * 4 : kNowhere, (row * ld + first) * 4, kPastL1));
            }
        }
#pragma unroll
        for (int u = 0; u < kRounds; ++u) {
            const int row = wave + u * kPresentWaves;
            if (row >= R) break;
            uint32_t q[RC];
            float scale;
            if constexpr (decltype(norm)::value)
                scale = panel_norm_quantize<EVEN>(v[u], c, PanelAffine<RC>(c, gamma, beta), p.eps, q);
            else
                scale = row_range_quantize<EVEN>(v[u], c, q);
            if (lane == 0) row_scale[row] = scale;
            uint32_t *dword = reinterpret_cast<uint32_t *>(codes);
#pragma unroll
            for (int i = 0; i < RC; ++i)
                if (c.real[i]) dword[((c.block[i] * 2 + c.part / 4) * kPiece + row) * 4 + c.part % 4] = q[i];
        }
        __syncthreads();
    };
    // The same of GELU's results.
    auto hidden_codes = [&] {
#pragma unroll 1
        for (int row = wave; row < R; row += kPresentWaves) {
            v4i raw[HC];
#pragma unroll
            for (int i = 0; i < HC; ++i) {
                const int col = 4 * (lane + kWave * i);
                raw[i] = __builtin_amdgcn_raw_buffer_load_b128(rqkv, col < d_ff && col < 3 * d ? (row * 3 * d + col) * 4 : kNowhere, 0, kPastL1);
                if (256 * i + 256 > 3 * d)  // (one of the two is out of range, which reads as zeros)
                    raw[i] |= __builtin_amdgcn_raw_buffer_load_b128(
                        rbeside, col < d_ff && col >= 3 * d ? (row * beside + col - 3 * d) * 4 : kNowhere, 0, kPastL1);
            }
            auto value = [&](int i, int e) {
                const int bits = raw[i][e];
                return __builtin_bit_cast(float, bits);
            };
            float am = 0.0f;  // (a NaN is no maximum)
#pragma unroll
            for (int i = 0; i < HC; ++i)
                am = fmaxf(am, fmaxf(fmaxf(fabsf(value(i, 0)), fabsf(value(i, 1))), fmaxf(fabsf(value(i, 2)), fabsf(value(i, 3)))));
            am = wave_max(am);
            const float scale = am < FLT_EPSILON ? 1.0f : am / 127.0f, inv = recip_for_div(scale);
            const bool good = am <= FLT_MAX;
            if (lane == 0) row_scale[row] = good ? scale : NAN;
            uint32_t *dword = reinterpret_cast<uint32_t *>(codes);
#pragma unroll
            for (int i = 0; i < HC; ++i) {
                const int col = 4 * (lane + kWave * i);
                if (col < d_ff)
                    dword[(col / 16 * kPiece + row) * 4 + col % 16 / 4] =
                        good ? pack4(quantize_int_sym<EVEN>(value(i, 0), scale, inv), quantize_int_sym<EVEN>(value(i, 1), scale, inv),
                                     quantize_int_sym<EVEN>(value(i, 2), scale, inv), quantize_int_sym<EVEN>(value(i, 3), scale, inv))
                             : 0u;
            }
        }
        __syncthreads();
    };
    auto product = [&](const int8_t *w, const float *scales, const float *biases, int nblocks, int kblocks, auto use) {
        const __amdgpu_buffer_rsrc_t rw = team_buffer(w, nblocks * kblocks * 1024);
        const int fragment = lane / 16 * 512 + lane % 16 * 16;
#pragma unroll 1
        for (int half = wave * members + rank; half < 2 * nblocks; half += members * kPresentWaves) {
            v4i acc{0, 0, 0, 0};
            const int n = half * 16 + lane % 16, from = half / 2 * kblocks * 1024 + half % 2 * 256;
            const float sw = scales[n], bias = biases ? biases[n] : 0.0f;
#pragma unroll 1
            for (int kb0 = 0; kb0 < kblocks; kb0 += 2 * kPresentChunk) {
                v4i fw[kPresentChunk];
#pragma unroll
                for (int u = 0; u < kPresentChunk; ++u)
                    if (kb0 + 2 * u < kblocks)
                        fw[u] = __builtin_amdgcn_raw_buffer_load_b128(rw, fragment, from + (kb0 + 2 * u) * 1024, 0);
#pragma unroll
                for (int u = 0; u < kPresentChunk; ++u)
                    if (kb0 + 2 * u < kblocks)
                        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(codes[((kb0 + 2 * u) * 2 + lane / 16) * kPiece + lane % kTeamRows], fw[u], acc, 0, 0, 0);
            }
            float o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                o[i] = static_cast<float>(acc[i]) * (row_scale[mine + i] * sw);
                o[i] = o[i] + bias;
            }
            use(half, n, o);
        }
        acknowledged();
    };
    auto store = [&](float v, const __amdgpu_buffer_rsrc_t &to, int at, int i) {  // result i of this lane, if its row is one of the team's
        if (mine + i < R) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), to, at * 4, 0, 0);
    };
    auto add_to_stream = [&](int, int n, float(&o)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int at = (mine + i) * d + n;
            const float x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, mine + i < R ? at * 4 : kNowhere, 0, kPastL1));
            store(o[i] + x, rx, at, i);
        }
    };
#pragma unroll 1
    for (int l = 0; l < p.layers; ++l) {
        const hipq_block_weights &b = p.blocks[l];
        if (l > 0 || !p.qkv_done) {
            row_codes(std::true_type{}, rx, d, 0, b.ln1_gamma, b.ln1_beta);
            product(b.w_qkv, b.s_qkv, b.b_qkv, 3 * dblocks, dblocks, [&](int, int n, float(&o)[4]) {
#pragma unroll
                for (int i = 0; i < 4; ++i) store(o[i], rqkv, (mine + i) * 3 * d + n, i);
            });
            meet();
        }
        row_codes(std::false_type{}, rqkv, 3 * d, 2 * d, nullptr, nullptr);
        product(b.w_out, b.s_out, b.b_out, dblocks, dblocks, add_to_stream);
        meet();
        row_codes(std::true_type{}, rx, d, 0, b.ln2_gamma, b.ln2_beta);
        product(b.w_fc1, b.s_fc1, b.b_fc1, fblocks, dblocks, [&](int half, int n, float(&o)[4]) {
            const bool in_rows = half * 16 < 3 * d;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float h = gelu_tanh(o[i]);
                if (in_rows)
                    store(h, rqkv, (mine + i) * 3 * d + n, i);
                else
                    store(h, rbeside, (mine + i) * beside + n - 3 * d, i);
            }
        });
        meet();
        hidden_codes();
        product(b.w_fc2, b.s_fc2, b.b_fc2, dblocks, fblocks, add_to_stream);
        if (l + 1 < p.layers) meet();
    }
    if (wave == 0 && lane == 0 && lost) __hip_atomic_store(p.wait_error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void team_words_clear_kernel(uint32_t *words) { words[blockIdx.x * blockDim.x + threadIdx.x] = 0; }

}  // namespace

// Up to 128 tokens of rows of up to 768 floats (16 rows a team, three float4 a lane).  Separate kernels / this, us: 12 layers of d 768,
// d_ff 3072 1 token 303 / 191, 16 313 / 217, 77 334 / 240, 128 368 / 281; d 384, d_ff 1152, 10 layers, 3 tokens 231 / 118; d 256,
// d_ff 1024, 6 layers, 40 tokens 140 / 82.  What is left is 2.3 us a phase (rows 0.5, LayerNorm and codes 1.1, product 0.3, results
// and their acknowledgement 0.9, meeting 0.35) and, at d 768, 7 MB of weights a layer through each XCD's port, at some 0.7 TB/s.
// Rows of up to 1024 floats would need three steps of K times three column blocks of weights in the registers of a wave that multiplies,
// where there is room for eight (115 of 128 are taken), or eight such waves and eight for the rows: not tried.
bool team_stack_fits(const hipq_ctx *ctx, const float *x, size_t tokens, size_t d, size_t d_ff, PanelFold after_out,
                     PanelFold after_fc2) {
    const int share = ctx->resident_share > 0 ? ctx->resident_share : 1;
    auto folds = [](PanelFold f) { return !f.pair && f.wave_blocks == kTeamFloats; };
    return ctx->pair_ok && share == 1 && ctx->num_cus >= kTeams * kTeamSize && folds(after_out) && folds(after_fc2) &&
           tokens <= kTeamTokens && d % 128 == 0 && d <= size_t(kTeamFloats) * 256 && d_ff % 128 == 0 &&
           d_ff <= size_t(kTeamColumns) * kTeamSize * 32 && d_ff <= 4 * d && (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
}

int32_t team_stack(hipq_ctx *ctx, const TeamStackCall &call, int32_t mode) {
    StackTeam p;
    p.x = call.x;
    p.qkv = call.qkv;
    p.maxima = call.maxima;
    p.codes = call.codes;
    p.words = call.words ? call.words : ctx->wait_error + kCtxTeamWord;
    if (call.words) hipLaunchKernelGGL(team_words_clear_kernel, dim3(kTeams), dim3(kCtxTeamWords), 0, ctx->stream, call.words);
    p.wait_error = ctx->wait_error;
    p.tokens = static_cast<int>(call.tokens);
    p.rows = static_cast<int>((call.tokens + kTeams - 1) / kTeams);
    p.d = static_cast<int>(call.d);
    p.d_ff = static_cast<int>(call.d_ff);
    p.spin_limit = ctx->wait_spin_limit < 1024 ? 1 << 20 : ctx->wait_spin_limit;  // (a small one, a test's, is for the assembly)
    p.assembly_limit = ctx->wait_spin_limit < kAssemblyLimit ? ctx->wait_spin_limit : kAssemblyLimit;
    p.gather_looks = ctx->wait_spin_limit == 0 ? 0 : kGatherLooks;
    p.eps = call.eps;
    for (size_t l = 0; l < call.layers; l += kTeamLayers) {
        p.layers = static_cast<int>(call.layers - l < size_t(kTeamLayers) ? call.layers - l : size_t(kTeamLayers));
        p.qkv_done = l == 0;
        for (int i = 0; i < p.layers; ++i) p.blocks[i] = call.blocks[l + i];
        if (mode & HIPQ_ROUND_HALF_EVEN) {
            hipLaunchKernelGGL(stack_team_kernel<true>, dim3(kTeams * kTeamSize), dim3(1024), 0, ctx->stream, p);
            hipLaunchKernelGGL(stack_present_kernel<true>, dim3(kTeams * kTeamSize), dim3(kPresentWaves * kWave), 0, ctx->stream, p);
        } else {
            hipLaunchKernelGGL(stack_team_kernel<false>, dim3(kTeams * kTeamSize), dim3(1024), 0, ctx->stream, p);
            hipLaunchKernelGGL(stack_present_kernel<false>, dim3(kTeams * kTeamSize), dim3(kPresentWaves * kWave), 0, ctx->stream, p);
        }
        const int32_t rc = check_launch("transformer stack (teams)");
        if (rc) return rc;
    }
    return HIPQ_SUCCESS;
}

}  // namespace hipq
