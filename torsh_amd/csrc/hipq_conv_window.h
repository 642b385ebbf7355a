// Quantized Conv2d of any stride and any channel count as an implicit GEMM on the matrix cores: rows of the product
// are the output positions ("windows", in output order: no padded grid), columns the output channels.
//
// Image layout.  The u8 NCHW input is rewritten once as signed bytes (x - 128) in
//   [channel group][image][padded row][padded pixel][pitch]
// with the channels cut into ceil(C / 32) groups of `pitch` bytes (the group's channels, rounded up to 4) and a border
// of the zero point.  One row of a filter's taps then covers kw * pitch CONSECUTIVE bytes, whatever the stride, so K is
// cut into k blocks of 32 bytes along (tap row, 32-byte piece of the row, channel group): a window's slice of a k block
// is two 16-byte pieces at (address of its first pixel) + (an offset that is the same for every window), which is
// exactly what a lane of v_mfma_i32_32x32x32_i8 holds.  A wave loads 32 windows' slice with one instruction whose
// per-lane offset never changes and whose k block is a scalar: no im2col, no gather, no LDS.  Windows overlap in
// memory; the vector-memory path and L1 see that, HBM does not.  Three channels (pitch 4, 7 taps: 28 of 32 bytes
// used) waste an eighth of the multiply, 32 channels nothing.  What a slice reads beyond its row of taps are other
// pixels' bytes; the packed filters hold zeros there.
//
// The filters are packed in the fragment order of hipq_gemm_packed.h with the same K order, and
// sum (x - zp) w = sum (x - 128) w + (128 - zp) sum w is undone per output channel in the epilogue.
//
// Measured against what it replaced, u8 in, filters as rows (us per forward): [32,3,224,224] x [64,3,7,7] stride 2
// 2288 -> 25.5 (a thread per output); [32,64,56,56] x [64,64,3,3] 63 -> 20, [32,128,28,28] x [128,128,3,3] 26.4 -> 17.6,
// [32,256,14,14] x [256,256,3,3] 20.9 -> 16.2, [32,512,7,7] x [512,512,3,3] 28.0 -> 23.5, [32,256,56,56] x [64,256,1,1] 50 -> 22
// (the packed GEMM over the padded grid, which always split K: its 128 x 64 tiles spend more on the sum of the partial
// products than on short K, compute the windows of the border, and store single bytes).  What bounds it now: at long K
// the vector-memory path, 6 KiB per 8 MFMAs; at short K (the first layer) instruction issue, 815 vector instructions per wave
// of which most are the requantize of its 64 x 64 outputs, and the misaligned 16-byte pieces (21.7 L1 accesses per load on
// average, 16 where they are a contiguous KiB).
//
// Waves.  A workgroup's four waves either take different windows (SPLIT = false: FM x FN accumulator blocks each, the
// filters' fragments coming out of L1 for three of the four) or split K and sum through LDS (SPLIT = true), which keeps
// all SIMDs busy when there are fewer tiles than that; or eight waves split the K of one block, for few windows, where
// latency is what counts.  A lane of the accumulators holds ONE output channel and 16
// windows: its scale, bias and zero-point correction are one register each, and after one exchange between the halves
// of the wave it owns 16 consecutive outputs of a channel's plane: one 16-byte store.
#pragma once

#include <type_traits>

#include "hipq_gemm_kernels.h"

namespace hipq {

struct ConvWindow {
    int M, N;             // output channels; windows = images * ho * wo
    int KB, kblocks;      // k blocks per filter row block as stored; those that hold data
    int cgs, segs;        // channel groups; 32-byte pieces per row of taps
    int pitch;            // bytes per pixel and channel group
    int row_bytes;        // wp * pitch
    int plane_bytes;      // bytes per channel group (nb * hp * wp * pitch)
    int image_bytes;      // cgs * plane_bytes
    int hp, wp, sh, sw, ho, wo;
    FastDiv by_plane, by_wo;  // window -> (image, position), position -> (row, column)
    FastDiv by_cgs, by_segs;  // k block -> (piece of all tap rows, channel group), -> (tap row, piece)
};

// 16, 4 x 4 and 4 bytes at an address that need not be aligned (global memory takes it; the outputs of a channel's plane
// start wherever ho * wo puts them).
struct __attribute__((packed, aligned(1))) ConvBytes16 {
    v4i v;
};
struct __attribute__((packed, aligned(4))) ConvWords4 {
    v4i v;
};
struct __attribute__((packed, aligned(1))) ConvWord {
    uint32_t v;
};

// u8 NCHW -> the layout above.  One thread per (channel group, V consecutive padded pixels of a row), DW dwords of four
// channels each (consecutive lanes are consecutive pixels: consecutive bytes of every channel plane).  V = 4: a channel's
// four pixels are one dword at any alignment, loaded from inside the image row and shifted where the run reaches over
// its end, and 4 x 4 bytes are transposed by eight permutes: a quarter of the loads and of the address arithmetic, which
// is what bounded the pass ([32,3,224,224] pad 3: 11.1 -> 5.5 us, filters included; 12 MB moved).  V = 1: groups
// of more than four channels that are all there (FULL: the loads of a pixel need no guard, and its bytes are one run of
// stores), rows of fewer than four pixels, images without rows.
// Further workgroups pack the filters: one output channel each, a thread per 16-byte piece.
struct ConvWindowFilters {
    const int8_t *w;  // [OC, IC, KH, KW]
    int8_t *packed;
    int32_t *wsum;
    int ic, kh, kw;
};

// How the image part of the grid is walked: runs of V pixels, `runs` to a padded row.
struct ConvPackWalk {
    int filters;        // workgroups that pack filters, ahead of the image's
    int groups_per_cg;  // workgroups per channel group
    int items;          // runs per channel group
    FastDiv by_runs, by_hp;
};

template <int DW, int V, bool FULL>
__global__ __launch_bounds__(256) void conv_window_pack_kernel(const uint8_t *__restrict__ x, int C, int H, int W, int pad_h,
                                                                 int pad_w, int zp, const int32_t *__restrict__ zp_dev,
                                                                 ConvPackWalk walk, int8_t *__restrict__ image,
                                                                 ConvWindow cw, ConvWindowFilters f) {
    static_assert(V == 1 || (V == 4 && !FULL), "pixels per thread");
    // The filters' workgroups come first: their chain (16 gathered bytes, a sum over the workgroup) is the longer one.
    if (static_cast<int>(blockIdx.x) < walk.filters) {
        __shared__ int part[4];
        const int oc = blockIdx.x, taps = f.kh * f.kw;
        const int8_t *w = f.w + size_t(oc) * f.ic * taps;
        int sum = 0;
        for (int piece = threadIdx.x; piece < cw.KB * 2; piece += 256) {
            const int kb = piece / 2, half = piece % 2;
            const int cg = kb % cw.cgs, seg = (kb / cw.cgs) % cw.segs, ty = kb / (cw.cgs * cw.segs);
            const int p = seg * 32 + half * 16;  // byte within the row of taps
            int tx = p / cw.pitch, c = p % cw.pitch;
            // All 16 requested before the first is used; a byte that is not a weight reads the first one and counts 0.
            int8_t v[16];
            bool real[16];
#pragma unroll
            for (int b = 0; b < 16; ++b) {
                const int ch = cg * cw.pitch + c;
                real[b] = kb < cw.kblocks && tx < f.kw && ch < f.ic;
                v[b] = w[real[b] ? ch * taps + ty * f.kw + tx : 0];
                if (++c == cw.pitch) {
                    c = 0;
                    ++tx;
                }
            }
            uint32_t d[4] = {0, 0, 0, 0};
#pragma unroll
            for (int b = 0; b < 16; ++b) {
                const int value = real[b] ? v[b] : 0;
                sum += value;
                d[b / 4] |= static_cast<uint32_t>(static_cast<uint8_t>(value)) << (8 * (b % 4));
            }
            *reinterpret_cast<uint4 *>(f.packed + (size_t(oc / 32) * cw.KB + kb) * 1024 + (oc % 32 + 32 * half) * 16) =
                make_uint4(d[0], d[1], d[2], d[3]);
        }
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, kWave);
        if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = sum;
        __syncthreads();
        if (threadIdx.x == 0) f.wsum[oc] = part[0] + part[1] + part[2] + part[3];
        return;
    }
    const int block = blockIdx.x - walk.filters, groups_per_cg = walk.groups_per_cg;
    if (zp_dev) zp = *zp_dev;  // the zero point a dynamic quantize has left on the device
    const int cg = block / groups_per_cg;
    const int item = (block % groups_per_cg) * 256 + threadIdx.x;
    if (item >= walk.items) return;
    uint32_t run, row;
    const uint32_t line = walk.by_runs.quotient(item, &run);  // padded row of the whole batch
    const uint32_t n = walk.by_hp.quotient(line, &row);
    const int h = static_cast<int>(row) - pad_h, v = static_cast<int>(run) * V - pad_w;
    const int pixels = cw.wp - static_cast<int>(run) * V < V ? cw.wp - static_cast<int>(run) * V : V;
    const uint32_t border = static_cast<uint32_t>(static_cast<uint8_t>(zp ^ 0x80)) * 0x01010101u;
    const size_t plane = size_t(H) * W;
    const int c0 = cg * DW * 4;
    uint32_t d[V][DW];
    if constexpr (V == 1) {
#pragma unroll
        for (int i = 0; i < DW; ++i) d[0][i] = border;
        if (h >= 0 && h < H && v >= 0 && v < W) {
            const uint8_t *src = x + ((size_t(n) * C + c0) * H + h) * W + v;
            uint32_t b[4 * DW];
#pragma unroll
            for (int c = 0; c < 4 * DW; ++c) b[c] = FULL || c0 + c < C ? src[size_t(c) * plane] : 0u;
#pragma unroll
            for (int i = 0; i < DW; ++i)
                d[0][i] = (b[4 * i] | (b[4 * i + 1] << 8) | (b[4 * i + 2] << 16) | (b[4 * i + 3] << 24)) ^ 0x80808080u;
        }
    } else {
        // The run's pixels v .. v + 3 from the dword at `at`, which lies inside the image row (W >= 4).
        const int hc = h < 0 ? 0 : (h < H ? h : H - 1);
        const int at = v < 0 ? 0 : (v < W - 4 ? v : W - 4);
        const uint8_t *src = x + ((size_t(n) * C + c0) * H + hc) * W + at;
        uint32_t b[4 * DW];
#pragma unroll
        for (int c = 0; c < 4 * DW; ++c) b[c] = c0 + c < C ? reinterpret_cast<const ConvWord *>(src + size_t(c) * plane)->v : 0u;
        const uint32_t left = 8 * (at - v), right = 8 * (v - at);  // one of them 0; from 32 on no pixel is inside
#pragma unroll
        for (int c = 0; c < 4 * DW; ++c) b[c] = v < at ? b[c] << (left & 31) : b[c] >> (right & 31);
        bool inside[V];
#pragma unroll
        for (int p = 0; p < V; ++p) inside[p] = h == hc && v + p >= 0 && v + p < W;
#pragma unroll
        for (int i = 0; i < DW; ++i) {
            const uint32_t lo0 = __builtin_amdgcn_perm(b[4 * i + 1], b[4 * i], 0x05010400u);  // c0p0 c1p0 c0p1 c1p1
            const uint32_t lo1 = __builtin_amdgcn_perm(b[4 * i + 1], b[4 * i], 0x07030602u);  // ... p2, p3
            const uint32_t hi0 = __builtin_amdgcn_perm(b[4 * i + 3], b[4 * i + 2], 0x05010400u);
            const uint32_t hi1 = __builtin_amdgcn_perm(b[4 * i + 3], b[4 * i + 2], 0x07030602u);
            const uint32_t t[4] = {__builtin_amdgcn_perm(hi0, lo0, 0x05040100u), __builtin_amdgcn_perm(hi0, lo0, 0x07060302u),
                                   __builtin_amdgcn_perm(hi1, lo1, 0x05040100u), __builtin_amdgcn_perm(hi1, lo1, 0x07060302u)};
#pragma unroll
            for (int p = 0; p < V; ++p) d[p][i] = inside[p] ? t[p] ^ 0x80808080u : border;
        }
    }
    uint32_t *dst = reinterpret_cast<uint32_t *>(image + size_t(cg) * cw.plane_bytes +
                                                 (size_t(line) * cw.wp + size_t(run) * V) * (4 * DW));
    if constexpr (V == 4 && DW == 1) {
        if (pixels == V) {
            reinterpret_cast<ConvWords4 *>(dst)->v = v4i{static_cast<int>(d[0][0]), static_cast<int>(d[1][0]),
                                                         static_cast<int>(d[2][0]), static_cast<int>(d[3][0])};
            return;
        }
    }
#pragma unroll
    for (int p = 0; p < V; ++p) {
        if (p >= pixels) break;
        if constexpr (DW % 4 == 0) {
#pragma unroll
            for (int i = 0; i < DW; i += 4)
                *reinterpret_cast<uint4 *>(dst + p * DW + i) = make_uint4(d[p][i], d[p][i + 1], d[p][i + 2], d[p][i + 3]);
        } else {
#pragma unroll
            for (int i = 0; i < DW; ++i) dst[p * DW + i] = d[p][i];
        }
    }
}

// Waves of a workgroup: four, or eight where they share the K of one accumulator block.
template <int FM, int FN, bool SPLIT>
constexpr int conv_window_waves = SPLIT && FM * FN == 1 ? 8 : 4;

template <int FM, int FN, int D, bool SPLIT, int EPI, bool EVEN>
__global__ __launch_bounds__((64 * conv_window_waves<FM, FN, SPLIT>),
                             FM * FN == 1 ? 2 : FM * FN < 8 ? 3 : (SPLIT ? 1 : 2)) void conv_i8_window_kernel(const int8_t *__restrict__ filters,
                                                               const int8_t *__restrict__ image, ConvWindow cw,
                                                               GemmEpilogue ep) {
    constexpr int NBLK = FM * FN;
    constexpr int WAVES = conv_window_waves<FM, FN, SPLIT>;
    constexpr bool ONE = WAVES == 8;  // (wave 0 finishes the block)
    constexpr int OWN = SPLIT && !ONE ? NBLK / 4 : NBLK;  // accumulator blocks a wave finishes
    static_assert(!SPLIT || ONE || (FM == 4 && FN == 2) || (FM == 2 && FN == 2) || (FM == 1 && FN == 4), "K-split tiles");
    constexpr int COLS = SPLIT ? 1 : FM;          // channel blocks among them
    extern __shared__ __attribute__((aligned(16))) int8_t lds[];
    const int lane = threadIdx.x % kWave, half = lane / 32;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int plane = cw.ho * cw.wo;
    // An XCD (workgroups b, b + 8, ...) takes a contiguous run of windows and, inside it, all channel tiles of a
    // window tile one after the other: the image rows are fetched into its L2 once.
    constexpr int kTileN = (SPLIT ? 1 : 4) * FN * 32;
    const int tiles_m = ((cw.M + 31) / 32 + FM - 1) / FM, tiles_n = (cw.N + kTileN - 1) / kTileN;
    const int per_xcd = (tiles_n + 7) / 8, slot = blockIdx.x / 8;
    const int tile_m = slot % tiles_m, tile_n = static_cast<int>(blockIdx.x % 8) * per_xcd + slot / tiles_m;
    if (slot / tiles_m >= per_xcd || tile_n >= tiles_n) return;
    const int q0 = tile_n * kTileN + (SPLIT ? 0 : wave * FN * 32);  // first window of this wave
    const int rb0 = tile_m * FM;

    // K-split: a wave numbers the tile's blocks by exclusive or with its own place, so that the blocks it will own after
    // the sum are its first ones and block b goes to wave `wave ^ (b / OWN)`: every wave runs the same code on the same
    // registers, no wave-dependent choice behind the main loop.
    const int jx = !SPLIT || ONE ? 0 : FM == 4 ? wave : FM == 2 ? wave >> 1 : 0;
    const int ix = !SPLIT || ONE ? 0 : FM == 4 ? 0 : FM == 2 ? wave & 1 : wave;
    // Operands of the epilogue, ahead of the main loop: one channel per lane and channel block.
    int corr[COLS];
    float sc[COLS], bias[COLS];
#pragma unroll
    for (int j = 0; j < COLS; ++j) {
        const int oc = (rb0 + (j ^ jx)) * 32 + lane % 32;
        const int occ = oc < cw.M ? oc : cw.M - 1;
        corr[j] = (ep.cv_zp_in ? 128 - *ep.cv_zp_in : ep.cv_corr_mul) * ep.cv_wsum[occ];
        sc[j] = 1.0f;
        bias[j] = -0.0f;  // (v + -0.0f is v, bit for bit)
        if constexpr (EPI != EPI_I32) {
            sc[j] = (ep.sa ? ep.sa[0] : ep.sa_scalar) * ep.sw[occ];
            if (ep.bias) bias[j] = ep.bias[occ];
        }
    }

    const __amdgpu_buffer_rsrc_t rf = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t *>(filters), 0, ((cw.M + 31) / 32) * cw.KB * 1024, 0x00020000);
    const __amdgpu_buffer_rsrc_t ri =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(image), 0, cw.image_bytes, 0x00020000);
    int sof[FM];
#pragma unroll
    for (int j = 0; j < FM; ++j) {
        int rb = rb0 + (j ^ jx);
        rb = rb < (cw.M + 31) / 32 ? rb : (cw.M + 31) / 32 - 1;  // (repeated: not stored)
        sof[j] = rb * cw.KB * 1024;
    }
    int voi[FN];
#pragma unroll
    for (int i = 0; i < FN; ++i) {
        int q = q0 + (i ^ ix) * 32 + lane % 32;
        q = q < cw.N ? q : cw.N - 1;
        uint32_t rem, ow;
        const uint32_t n = cw.by_plane.quotient(q, &rem), oh = cw.by_wo.quotient(rem, &ow);
        voi[i] = ((n * cw.hp + oh * cw.sh) * cw.wp + ow * cw.sw) * cw.pitch + 16 * half;
    }
    // This wave's next k block as (tap row, piece, channel group) and its offset in the image.  Steps of eight are divided,
    // not counted: with one channel group (images of up to 32 channels) counting is eight turns of the loop for every step
    // ahead of the first loads, us from u8 [4,32,28,28] x [128,32,1,1] 10.7 -> 8.5, [1,32,56,56] x [64,32,3,3] 9.0 -> 8.1.
    constexpr int STEP = SPLIT ? WAVES : 1;
    int kb = 0, cg = 0, seg = 0, ty = 0;
    auto advance = [&](int by) {
        kb += by;
        if constexpr (ONE) {
            uint32_t g, t;
            ty = cw.by_segs.quotient(cw.by_cgs.quotient(kb, &g), &t);
            cg = g;
            seg = t;
            return;
        }
        cg += by;
        while (cg >= cw.cgs) {
            cg -= cw.cgs;
            if (++seg == cw.segs) {
                seg = 0;
                ++ty;
            }
        }
    };
    if constexpr (SPLIT) advance(wave);
    v4i ff[D][FM], fi[D][FN];
    auto issue = [&](int s) {
        // A k block past the last: the filters' load lies beyond its buffer (zeros, no memory access), so what the windows
        // bring does not count: the first k block's.
        const bool real = kb < cw.kblocks;
        const int vof = real ? lane * 16 : 0x7fffffff;
        const int kof = real ? kb * 1024 : 0;
        const int koi = real ? cg * cw.plane_bytes + ty * cw.row_bytes + seg * 32 : 0;
#pragma unroll
        for (int j = 0; j < FM; ++j)
            ff[s][j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rf, vof, real ? sof[j] + kof : 0, 0));
#pragma unroll
        for (int i = 0; i < FN; ++i)
            fi[s][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(ri, voi[i], koi, 0));
        advance(STEP);
    };
    v16i acc[FM][FN];
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[j][i][r] = SPLIT ? 0 : corr[j];
    auto compute = [&](int s) {
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
            for (int i = 0; i < FN; ++i)
                acc[j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fi[s][i], ff[s][j], acc[j][i], 0, 0, 0);
    };
    const int steps = (cw.kblocks + STEP - 1) / STEP, rounds_end = (steps + D - 1) / D * D;
#pragma unroll
    for (int u = 0; u < D; ++u) issue(u);
    for (int s0 = D; s0 < rounds_end; s0 += D) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            compute(u);
            issue(u);
        }
    }
#pragma unroll
    for (int u = 0; u < D; ++u) compute(u);

    // Outputs of one accumulator block: channel block column j of this wave's constants, first window q.
    const float zpf = static_cast<float>(ep.zp_out);
    const uint32_t offset2 = static_cast<uint32_t>(ep.zp_out + 128) * 0x10001u;
    RequantFast fast[COLS];
    auto emit_block = [&](const v16i &a, int j, int oc, int q, auto plain) {
        auto dequant = [&](int r) { return static_cast<float>(a[r]) * sc[j] + bias[j]; };
        if constexpr (EPI == EPI_I8) {
            // register 4 g + i of half h is window 8 g + 4 h + i; after the exchange half h holds windows 16 h .. + 15
            uint32_t w[4];
            bool done = false;
            if constexpr (decltype(plain)::value) done = requant_fast16(a, fast[j], offset2, w);
            if (!done) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float v[4] = {dequant(4 * g), dequant(4 * g + 1), dequant(4 * g + 2), dequant(4 * g + 3)};
                    if constexpr (decltype(plain)::value) {
                        w[g] = requant_pack4<EVEN>(v, ep.s_out, ep.s_out_inv, offset2);
                    } else {
                        auto code = [&](float f) {  // NaN -> 0
                            return clamp_to_int(round_mode<EVEN>(div_rn(f, ep.s_out, ep.s_out_inv)) + zpf, -128, 127);
                        };
                        w[g] = pack4(code(v[0]), code(v[1]), code(v[2]), code(v[3]));
                    }
                }
            }
            const auto lo = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
            const auto hi = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
            const v4i bytes = {static_cast<int>(lo[0]), static_cast<int>(lo[1]), static_cast<int>(hi[0]),
                               static_cast<int>(hi[1])};
            const int first = q + 16 * half;
            if (oc >= cw.M || first >= cw.N) return;
            uint32_t pos;
            const uint32_t n = cw.by_plane.quotient(first, &pos);
            int8_t *o = static_cast<int8_t *>(ep.out) + (size_t(n) * cw.M + oc) * plane + pos;
            if (static_cast<int>(pos) + 16 <= plane) {
                reinterpret_cast<ConvBytes16 *>(o)->v = bytes;
            } else {  // the run crosses into the next image (or the end)
                const size_t skip = size_t(cw.M - 1) * plane;  // from the end of this plane to the next image's
                int at = static_cast<int>(pos);
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    if (first + k < cw.N) *o = static_cast<int8_t>(bytes[k / 4] >> (8 * (k % 4)));
                    ++o;
                    if (++at == plane) {
                        at = 0;
                        o += skip;
                    }
                }
            }
        } else {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                auto bits = [&](int r) {
                    if constexpr (EPI == EPI_I32) return a[r];
                    return __builtin_bit_cast(int, dequant(r));
                };
                const v4i four = {bits(4 * g), bits(4 * g + 1), bits(4 * g + 2), bits(4 * g + 3)};
                const int first = q + 8 * g + 4 * half;
                if (oc >= cw.M || first >= cw.N) continue;
                uint32_t pos;
                const uint32_t n = cw.by_plane.quotient(first, &pos);
                int32_t *o = static_cast<int32_t *>(ep.out) + (size_t(n) * cw.M + oc) * plane + pos;
                if (static_cast<int>(pos) + 4 <= plane) {
                    reinterpret_cast<ConvWords4 *>(o)->v = four;
                } else {
                    const size_t skip = size_t(cw.M - 1) * plane;
                    int at = static_cast<int>(pos);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        if (first + k < cw.N) *o = four[k];
                        ++o;
                        if (++at == plane) {
                            at = 0;
                            o += skip;
                        }
                    }
                }
            }
        }
    };
    bool all_plain = ep.zp_out >= -32000 && ep.zp_out <= 32000;  // (zp + 128 has 16 bits in the packed clamp)
    if constexpr (EPI == EPI_I8) {
#pragma unroll
        for (int j = 0; j < COLS; ++j) fast[j] = RequantFast(sc[j], bias[j], ep.s_out_inv, ep.zp_out);
#pragma unroll
        for (int j = 0; j < COLS; ++j) all_plain = all_plain && requant_is_plain(sc[j], bias[j], ep.s_out_inv);
    }
    auto with_division = [&](auto finish) {
        if constexpr (EPI == EPI_I8) {
            if (!all_plain) return finish(std::false_type{});
        }
        finish(std::true_type{});
    };
    if constexpr (!SPLIT) {
        with_division([&](auto plain) {
#pragma unroll
            for (int j = 0; j < FM; ++j)
#pragma unroll
                for (int i = 0; i < FN; ++i)
                    if ((rb0 + j) * 32 < cw.M)  // (a channel block past the last has no outputs)
                        emit_block(acc[j][i], j, (rb0 + j) * 32 + lane % 32, q0 + i * 32, plain);
        });
    } else if constexpr (ONE) {
        v4i *red = reinterpret_cast<v4i *>(lds);  // [wave - 1][register quad][lane]
        if (wave > 0) {
#pragma unroll
            for (int g = 0; g < 4; ++g)
                red[((wave - 1) * 4 + g) * kWave + lane] =
                    v4i{acc[0][0][4 * g], acc[0][0][4 * g + 1], acc[0][0][4 * g + 2], acc[0][0][4 * g + 3]};
        }
        __syncthreads();
        if (wave > 0) return;
        v16i own;
#pragma unroll
        for (int r = 0; r < 16; ++r) own[r] = acc[0][0][r] + corr[0];
#pragma unroll
        for (int s = 0; s < WAVES - 1; ++s)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const v4i part = red[(s * 4 + g) * kWave + lane];
#pragma unroll
                for (int i = 0; i < 4; ++i) own[4 * g + i] += part[i];
            }
        with_division([&](auto plain) { emit_block(own, 0, rb0 * 32 + lane % 32, q0, plain); });
    } else {
        // Blocks OWN .. NBLK - 1 are other waves': parked in LDS as [owner][slot][register quad][lane].
        v4i *red = reinterpret_cast<v4i *>(lds);
#pragma unroll
        for (int b = OWN; b < NBLK; ++b) {
            const int owner = wave ^ (b / OWN);
            v4i *dst = red + (owner * (NBLK - OWN) + b - OWN) * 4 * kWave + lane;
#pragma unroll
            for (int g = 0; g < 4; ++g)
                dst[g * kWave] = v4i{acc[b / FN][b % FN][4 * g], acc[b / FN][b % FN][4 * g + 1],
                                     acc[b / FN][b % FN][4 * g + 2], acc[b / FN][b % FN][4 * g + 3]};
        }
        __syncthreads();
        // All reads first, then the adds.
        v4i part[3][OWN][4];
        const v4i *src = red + wave * (NBLK - OWN) * 4 * kWave + lane;
#pragma unroll
        for (int s = 0; s < 3; ++s)
#pragma unroll
            for (int k = 0; k < OWN; ++k)
#pragma unroll
                for (int g = 0; g < 4; ++g) part[s][k][g] = src[((s * OWN + k) * 4 + g) * kWave];
        __builtin_amdgcn_sched_barrier(0);
        v16i own[OWN];
#pragma unroll
        for (int k = 0; k < OWN; ++k)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                own[k][r] = acc[0][k][r] + corr[0] + part[0][k][r / 4][r % 4] + part[1][k][r / 4][r % 4] + part[2][k][r / 4][r % 4];
        with_division([&](auto plain) {
#pragma unroll
            for (int k = 0; k < OWN; ++k)
                emit_block(own[k], 0, (rb0 + jx) * 32 + lane % 32, q0 + (k ^ ix) * 32, plain);
        });
    }
}

template <int FM, int FN, int D, bool SPLIT, int EPI, bool EVEN>
static int32_t launch_conv_window_form(hipq_ctx *ctx, const int8_t *filters, const int8_t *image, const ConvWindow &cw,
                                       const GemmEpilogue &ep) {
    constexpr int kWaves = conv_window_waves<FM, FN, SPLIT>;
    constexpr int kLds = SPLIT ? FM * FN * (kWaves - 1) * 4096 : 0;
    auto kernel = conv_i8_window_kernel<FM, FN, D, SPLIT, EPI, EVEN>;
    static bool configured[16] = {false};  // per device: raise the dynamic LDS limit once
    if (SPLIT && ctx->device < 16 && !configured[ctx->device]) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
        if (e != hipSuccess)
            return fail(HIPQ_DEVICE_ERROR, "conv2d: cannot reserve %d bytes of LDS: %s", kLds, hipGetErrorString(e));
        configured[ctx->device] = true;
    }
    constexpr int kTileN = (SPLIT ? 1 : 4) * FN * 32;
    const int tiles_m = ((cw.M + 31) / 32 + FM - 1) / FM, tiles_n = (cw.N + kTileN - 1) / kTileN;
    hipLaunchKernelGGL(kernel, dim3((tiles_n + 7) / 8 * 8 * tiles_m), dim3(64 * kWaves), kLds, ctx->stream, filters, image, cw, ep);
    return check_launch("conv2d (windows)");
}

}  // namespace hipq
