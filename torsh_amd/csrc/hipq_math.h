// Device-side scalar arithmetic of the quantized path.  Each helper states the
// Rust semantics it reproduces; the translation units are compiled with
// -ffp-contract=off so no multiply-add is fused and every f32 operation rounds
// exactly as the reference's CPU code does.
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

#include "torsh_hipq.h"

namespace hipq {

constexpr int kWave = 64;

// Waits until at most N of the wave's vector memory operations are under way.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    // gfx9 s_waitcnt encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] at [15:14]
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// Streaming (non-temporal) 16-byte and 4-byte accesses for data touched once.  Measured on
// MI355X over 16 Mi elements: quantize (64 MiB read, 16 MiB written) 19.8 us with ordinary
// accesses, 17.6 us with both streams non-temporal; dequantize (16 MiB read, 64 MiB written)
// 19.3 us ordinary, 13.4 us with ordinary loads and non-temporal stores (non-temporal loads
// of the small side cost 4 us there, so dequantize keeps ordinary loads).
typedef float hipq_vf4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 load_stream(const float4 *p) {
    const hipq_vf4 t = __builtin_nontemporal_load(reinterpret_cast<const hipq_vf4 *>(p));
    return make_float4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ uint32_t load_stream(const uint32_t *p) { return __builtin_nontemporal_load(p); }
__device__ __forceinline__ void store_stream(float4 *p, float4 v) {
    const hipq_vf4 t = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(t, reinterpret_cast<hipq_vf4 *>(p));
}
__device__ __forceinline__ void store_stream(uint32_t *p, uint32_t v) { __builtin_nontemporal_store(v, p); }

// Four floats at an address that is a multiple of four bytes only.
struct __attribute__((packed, aligned(4))) AnyFloat4 {
    float x, y, z, w;
};

// RND 0: f32::round (half away from zero); 1: IEEE nearest-even; 2: floor(v + 0.5), the
// "faster rounding" of quantize_mobile_optimized (crates/torsh-quantization/src/simd_ops.rs:426-428),
// with the f32 sum rounded before the floor as there.  Callers that know two modes pass a bool.
// Half away from zero as trunc(v + copysign(h, v)) with h the largest float below 0.5: three
// instructions (v_bfi, v_add, v_trunc) instead of the six of the library roundf.  With 0.5 itself
// the sum rounds up across an integer for v = +-0.49999997; with h it never does, and ties still
// land on the integer away from zero because v + h then rounds to even = that integer.  Checked
// against roundf for every finite float (tests/host/round_away_check.c).
template <int RND>
__device__ __forceinline__ float round_mode(float v) {
    if constexpr (RND == 1)
        return rintf(v);
    else if constexpr (RND == 2)
        return floorf(v + 0.5f);
    else
        return truncf(v + copysignf(0x1.fffffep-2f, v));
}

// f32::clamp: NaN passes through.
__device__ __forceinline__ float clamp_keep_nan(float v, float lo, float hi) {
    v = (v < lo) ? lo : v;
    v = (v > hi) ? hi : v;
    return v;
}

// `f32 as i32` on a value already clamped to a small range: NaN -> 0.
__device__ __forceinline__ int to_int_nan0(float v) { return (v != v) ? 0 : static_cast<int>(v); }

// `f32 as i32`, saturating, NaN -> 0.
__device__ __forceinline__ int f32_as_i32(float v) {
    if (v != v) return 0;
    if (v >= 2147483648.0f) return INT32_MAX;
    if (v <= -2147483648.0f) return INT32_MIN;
    return static_cast<int>(v);
}

// a / b, correctly rounded, from y = 1.0f / b (itself correctly rounded) with two FMAs
// (Markstein): q0 = RN(a*y), r = a - q0*b (exact in the FMA), q = RN(q0 + r*y).  Holds for every
// a while y is a normal number; an exhaustive CPU check over all 2^23 numerator significands x 22
// exponents x 3007 denominators (5.5e11 quotients) found no difference from a / b.  A division by
// one scale for a whole row or tensor then costs 3-4 instructions per element instead of the
// ~12 of the IEEE sequence.  y == 0 selects the plain division (recip_for_div returns 0 when
// 1/b is not normal); a NaN correction (a infinite, a quotient that overflows, NaN input) means q0
// already is the quotient.
__device__ __forceinline__ float recip_for_div(float b) {
    const float y = 1.0f / b;
    return (fabsf(y) >= FLT_MIN && fabsf(y) <= FLT_MAX) ? y : 0.0f;
}
__device__ __forceinline__ float div_rn(float a, float b, float y) {
    if (y == 0.0f) return a / b;
    const float q0 = a * y;
    const float r = fmaf(-q0, b, a);
    const float q1 = fmaf(r, y, q0);
    return (q1 == q1) ? q1 : q0;
}

// The reference's "quantize one value" formulas differ in where the zero point enters:
//   FORM 0  round(x * (1/scale)) + zp     crates/torsh-quantization/src/simd_ops.rs:36-46
//   FORM 1  round(x / scale) + zp         crates/torsh-quantization/src/algorithms.rs:230-233, 302-305
//   FORM 2  round(x / scale + zp)         crates/torsh-core/src/dtype/quantized.rs:129-134 (QInt8 / QUInt8)
//   FORM 3  (round(x / scale) as i32) + zp   crates/torsh-nn/src/quantization/ops.rs:153-162 (NaN -> 0 before zp)
// A bool first argument reads as FORM 0 / 1.  `inv` is recip_for_div(scale) for the division forms, else 1/scale.
enum { QFORM_MUL = 0, QFORM_DIV = 1, QFORM_DIV_ZP_FIRST = 2, QFORM_DIV_INT_CAST = 3 };

// Saturating f32 -> i32 with NaN -> 0: exactly Rust's `as i32`, and exactly what
// v_cvt_i32_f32 does.  Inline asm so the conversion is never treated as undefined for
// out-of-range inputs.
__device__ __forceinline__ int cvt_i32_sat(float v) {
    int r;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// The quantized value, clamped; result still a float (the carrier).
template <int FORM, int RND>
__device__ __forceinline__ float quantize_value(float x, float scale, float inv, float zpf, float lo, float hi) {
    float t;
    if constexpr (FORM != QFORM_MUL)
        t = div_rn(x, scale, inv);
    else
        t = x * inv;
    float q;
    if constexpr (FORM == QFORM_DIV_ZP_FIRST)
        q = round_mode<RND>(t + zpf);
    else if constexpr (FORM == QFORM_DIV_INT_CAST)
        q = static_cast<float>(cvt_i32_sat(round_mode<RND>(t))) + zpf;  // clamped to a small range next
    else
        q = round_mode<RND>(t) + zpf;
    return clamp_keep_nan(q, lo, hi);
}

// Integer form of quantize_value for int8/uint8 outputs: the clamp is done after the
// conversion, on integers (round(..)+zp is integral, so converting first changes nothing;
// a NaN becomes 0 as `NaN.clamp(..) as i8` does, and +-Inf saturate).  About half the
// vector instructions of the float-clamp form.
template <int FORM, int RND>
__device__ __forceinline__ int quantize_int(float x, float scale, float inv, float zpf, int lo, int hi) {
    float t;
    if constexpr (FORM != QFORM_MUL)
        t = div_rn(x, scale, inv);
    else
        t = x * inv;
    int q;
    if constexpr (FORM == QFORM_DIV_ZP_FIRST) {
        q = cvt_i32_sat(round_mode<RND>(t + zpf));
    } else if constexpr (FORM == QFORM_DIV_INT_CAST) {
        // i32 sum of the reference; the inner clamp keeps it from wrapping and changes nothing after the outer one
        q = min(max(cvt_i32_sat(round_mode<RND>(t)), -(1 << 30)), 1 << 30) + static_cast<int>(zpf);
    } else {
        q = cvt_i32_sat(round_mode<RND>(t) + zpf);
    }
    return min(max(q, lo), hi);
}

// FORM 3 with the zero point as the integer it is: (round(x / scale) as i32) + zp, the sum taken in 64 bits (the
// reference's i32 sum never wraps where it does not panic), then the clamp.  A constant channel of torsh-nn's
// per-channel weights has scale 0 and a zero point at an end of the i32 range, which a float cannot carry.
template <int RND>
__device__ __forceinline__ int quantize_int_cast(float x, float scale, float inv, int zp, int lo, int hi) {
    const long long q = static_cast<long long>(cvt_i32_sat(round_mode<RND>(div_rn(x, scale, inv)))) + zp;
    return static_cast<int>(q < lo ? lo : (q > hi ? hi : q));
}

// quantize_int for a symmetric per-row quantizer (zero point 0, int8 range) whose scale was derived
// from the row's own finite maximum, scale = max|x| / 127: then |x * y| stays near 127, the
// remainder of div_rn is never NaN for a finite x, and the select that guards it can go; a NaN
// element still comes out as 0 (NaN propagates through both FMAs and the conversion maps it to 0).
template <bool EVEN>
__device__ __forceinline__ int quantize_int_sym(float x, float scale, float y) {
    float t;
    if (y == 0.0f) {
        t = x / scale;
    } else {
        const float q0 = x * y;
        t = fmaf(fmaf(-q0, scale, x), y, q0);
    }
    return min(max(cvt_i32_sat(round_mode<EVEN>(t)), -128), 127);
}

// clamp(round(v) ...) already formed as a float: convert and clamp on integers.
__device__ __forceinline__ int clamp_to_int(float q, int lo, int hi) { return min(max(cvt_i32_sat(q), lo), hi); }

// Low bytes of four ints -> one dword (three v_perm_b32 / v_or).
__device__ __forceinline__ uint32_t pack4(int a, int b, int c, int d) {
    const uint32_t lo = __builtin_amdgcn_perm(static_cast<uint32_t>(b), static_cast<uint32_t>(a), 0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm(static_cast<uint32_t>(d), static_cast<uint32_t>(c), 0x04000c0cu);
    return lo | hi;
}

// Four bytes clamp(q + zp, -128, 127) in one dword; offset2 holds zp + 128 in both halves.  To i16 with saturation, +
// offset with saturation, to u8 with saturation, then the top bits flipped.
__device__ __forceinline__ uint32_t saturate_pack4(int q0, int q1, int q2, int q3, uint32_t offset2) {
    uint32_t h[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        uint32_t t;
        asm("v_cvt_pk_i16_i32 %0, %1, %2" : "=v"(t) : "v"(i ? q2 : q0), "v"(i ? q3 : q1));
        asm("v_pk_add_i16 %0, %1, %2 clamp" : "=v"(t) : "v"(t), "v"(offset2));
        asm("v_sat_pk_u8_i16 %0, %1" : "=v"(h[i]) : "v"(t));
    }
    return ((h[1] << 16) | h[0]) ^ 0x80808080u;
}
// Four requantized bytes clamp(round(v / s) + zp, -128, 127) in one dword, for values whose quotient is finite
// (requant_is_plain).  inv = recip_for_div(s), not 0; offset2 holds zp + 128 in both halves.  Division as div_rn
// without its guards; the clamp by the saturating packs: to i16, + offset saturating, to u8, then the top bits flipped
// (11 instructions per value where the guards and min / max per value made 18).
template <bool EVEN>
__device__ __forceinline__ uint32_t requant_pack4(const float (&v)[4], float s, float inv, uint32_t offset2) {
    int q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float q0 = v[i] * inv;
        const float d = fmaf(fmaf(-q0, s, v[i]), inv, q0);
        // v_cvt_i32_f32 truncates: the trunc of round_mode<0> is its own
        q[i] = cvt_i32_sat(EVEN ? rintf(d) : d + copysignf(0x1.fffffep-2f, d));
    }
    return saturate_pack4(q[0], q[1], q[2], q[3], offset2);
}
// The codes of 16 accumulators in one fused multiply-add each, where that is provably the same: with A = sc / s and
// B = bias / s + 1/2 + eps in f32, U = fma(acc, A, B) is within eps of (the quotient the exact chain rounds) + 1/2 + eps,
// so floor(U) is the code unless U lies less than 2 eps above an integer; which way ties go never matters.  With u = 2^-24,
// b = |bias / s| and |quotient| <= T: the chain's multiply, add and divide are off by u (T + b) + u T + u T, A by 2 u, B by
// 2 u b + u |B| and the fma by u |U|, together at most u (6 T + 6 b + 2); codes beyond T = 129 + |zp| saturate either way.
// A lane that has such a value (once in ten blocks of 1024 at T = 129) sends the wave to the exact form: 6.5 instructions
// per value instead of 11 where it does not.
struct RequantFast {
    float a, b, limit;
    __device__ __forceinline__ RequantFast() {}
    __device__ __forceinline__ RequantFast(float sc, float bias, float inv, int zp) {
        const float t = 129.0f + fabsf(static_cast<float>(zp)), bq = bias * inv;
        const float eps = (6.0f * t + 6.0f * fabsf(bq) + 4.0f) * 0x1.02p-24f;
        a = sc * inv;
        b = bq + (0.5f + eps);
        limit = 2.0f * eps;
    }
};
// w[g]: the bytes of accumulators 4 g .. 4 g + 3, valid where it returns true (the same for all lanes of the wave).
// For values that requant_is_plain has cleared.
template <typename Acc>
__device__ __forceinline__ bool requant_fast16(const Acc &acc, const RequantFast &f, uint32_t offset2, uint32_t (&w)[4]) {
    int q[16];
    float low = 1.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float v = fmaf(static_cast<float>(acc[r]), f.a, f.b);
        low = fminf(low, __builtin_amdgcn_fractf(v));
        asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(q[r]) : "v"(v));
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) w[g] = saturate_pack4(q[4 * g], q[4 * g + 1], q[4 * g + 2], q[4 * g + 3], offset2);
    return !__any(!(low >= f.limit));
}
// Whether requant_pack4 may take every value acc * scale + bias (|acc| < 2^31) of this wave.
__device__ __forceinline__ bool requant_is_plain(float scale, float bias, float inv) {
    const float most = (fabsf(scale) * 2147483648.0f + fabsf(bias)) * fabsf(inv);
    return inv != 0.0f && __all(most < 1e37f);
}

// 4 x 4 byte transpose inside a quad of lanes: lane q holds bytes (row 0..3) of column q and ends with the bytes
// (column 0..3) of row q.  Two butterfly steps - swap with lane q ^ 1 and interleave bytes, swap with lane q ^ 2 and
// interleave halves - each a data-parallel move and a byte permute whose selector depends on the lane:
// sel1 = q & 1 ? 0x03070105 : 0x06020400, sel2 = q & 2 ? 0x03020706 : 0x05040100.
__device__ __forceinline__ uint32_t quad_byte_transpose(uint32_t d, uint32_t sel1, uint32_t sel2) {
    const uint32_t p1 = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(d), 0xB1, 0xf, 0xf, true));
    const uint32_t t = __builtin_amdgcn_perm(p1, d, sel1);
    const uint32_t p2 = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(t), 0x4E, 0xf, 0xf, true));
    return __builtin_amdgcn_perm(p2, t, sel2);
}

// Butterfly over the 64 lanes in the order lane ^ 32, 16, 8, 4, 2, 1, all lanes ending with the result; op commutes.  The
// two wide steps are the half and the row swap, the others moves inside a row of 16: a rotation by 8, by 4 (equal to
// lane ^ 4, since lanes 8 apart agree by then) and two quad permutes.  A step is two dependent vector instructions instead
// of a trip through LDS, which is what a kernel of one row per wave waits for (LayerNorm + quantize of 77 x 768: three such
// reductions one after the other).
template <int CTRL>
__device__ __forceinline__ float lane_move(float v) {
    const int b = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(b, b, CTRL, 0xf, 0xf, true));
}
template <typename Op>
__device__ __forceinline__ float wave_butterfly(float v, Op op) {
    uint32_t b = __builtin_bit_cast(uint32_t, v);
    const auto halves = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    // (through scalars: a bit cast of a vector's element takes its first one)
    const uint32_t h0 = halves[0], h1 = halves[1];
    v = op(__builtin_bit_cast(float, h0), __builtin_bit_cast(float, h1));
    b = __builtin_bit_cast(uint32_t, v);
    const auto rows = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    const uint32_t r0 = rows[0], r1 = rows[1];
    v = op(__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1));
    v = op(v, lane_move<0x128>(v));  // row_ror:8
    v = op(v, lane_move<0x124>(v));  // row_ror:4
    v = op(v, lane_move<0x4E>(v));   // quad_perm [2, 3, 0, 1]
    return op(v, lane_move<0xB1>(v));  // quad_perm [1, 0, 3, 2]
}

// The sum over the 64 lanes folded in the order lane ^ 1, 2, 4, 8, 16, 32 (the mirrors of 8 and 16 lanes stand for ^ 4 and
// ^ 8: the lanes they combine agree inside the smaller groups by then).
__device__ __forceinline__ float wave_sum_ascending(float v) {
    v = v + lane_move<0xB1>(v);   // quad_perm [1, 0, 3, 2]
    v = v + lane_move<0x4E>(v);   // quad_perm [2, 3, 0, 1]
    v = v + lane_move<0x141>(v);  // row_half_mirror
    v = v + lane_move<0x140>(v);  // row_mirror
    uint32_t b = __builtin_bit_cast(uint32_t, v);
    const auto rows = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    const uint32_t r0 = rows[0], r1 = rows[1];
    v = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
    b = __builtin_bit_cast(uint32_t, v);
    const auto halves = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    const uint32_t h0 = halves[0], h1 = halves[1];
    return __builtin_bit_cast(float, h0) + __builtin_bit_cast(float, h1);
}

__device__ __forceinline__ float wave_min(float v) {
    return wave_butterfly(v, [](float a, float b) { return fminf(a, b); });
}

__device__ __forceinline__ float wave_max(float v) {
    return wave_butterfly(v, [](float a, float b) { return fmaxf(a, b); });
}

// n / d for 0 <= n < 2^31 by a multiply-high and a shift, where the compiler's division of a lane's value by a launch
// argument is some thirty instructions, a third of them at quarter rate.  With L = ceil(log2 d) the multiplier is
// m = floor(2^(31 + L) / d) + 1 <= 2^32 - 1, so m d = 2^(31 + L) + e with 0 < e <= d <= 2^L, and n m / 2^(31 + L)
// exceeds n / d by n e / (d 2^(31 + L)) < 1 / d: the floor is the quotient.
struct FastDiv {
    uint32_t d, m;
    int shift;
    __host__ static FastDiv by(uint32_t d) {  // 1 <= d < 2^31
        if (d <= 1) return FastDiv{1, 0, 0};
        int l = 0;
        while ((uint64_t(1) << l) < d) ++l;
        return FastDiv{d, static_cast<uint32_t>((uint64_t(1) << (31 + l)) / d + 1), l - 1};
    }
    __device__ __forceinline__ uint32_t quotient(uint32_t n) const { return d == 1 ? n : __umulhi(n, m) >> shift; }
    __device__ __forceinline__ uint32_t quotient(uint32_t n, uint32_t *rem) const {
        const uint32_t q = quotient(n);
        *rem = n - q * d;
        return q;
    }
};

// A kernel that writes a parameter record writes all of it, so that the record needs no fill before.
__device__ __forceinline__ void clear_reserved(hipq_qparams *p) {
#pragma unroll
    for (int i = 0; i < 3; ++i) p->reserved[i] = 0;
}

// (min,max) -> (scale, zero_point) with the reference formula `flavor` selects.
// Returns HIPQ_SUCCESS or HIPQ_INVALID_ARGUMENT.
//   HIPQ_PARAMS_SYMMETRIC          crates/torsh-quantization/src/algorithms.rs:397-422
//   HIPQ_PARAMS_AFFINE             crates/torsh-quantization/src/algorithms.rs:358-394
//   HIPQ_PARAMS_BACKEND_SYMMETRIC  crates/torsh-backend/src/quantization/params.rs:323-340
//   HIPQ_PARAMS_BACKEND_ASYMMETRIC crates/torsh-backend/src/quantization/params.rs:343-363
//   HIPQ_PARAMS_ZERO_INCLUDED      crates/torsh-quantization/src/observers.rs:263-310, specialized.rs:39-48, 322-335
//   HIPQ_PARAMS_NN_SYMMETRIC       crates/torsh-nn/src/quantization/ops.rs:322-325 (no guards: a zero range gives scale 0)
//   HIPQ_PARAMS_NN_ASYMMETRIC      crates/torsh-nn/src/quantization/ops.rs:326-330 (zero point not clamped)
__device__ __forceinline__ int params_from_minmax(float mn, float mx, int flavor, int qmin_i, int qmax_i,
                                                  float *scale, int *zp) {
    const bool finite = (fabsf(mn) <= FLT_MAX) && (fabsf(mx) <= FLT_MAX);  // false for NaN and Inf
    const float qmin = static_cast<float>(qmin_i), qmax = static_cast<float>(qmax_i);
    *scale = 1.0f;
    *zp = 0;
    switch (flavor) {
    case HIPQ_PARAMS_SYMMETRIC: {
        if (!finite) return HIPQ_INVALID_ARGUMENT;
        float abs_max = fmaxf(fabsf(mn), fabsf(mx));
        if (abs_max < FLT_EPSILON) return HIPQ_SUCCESS;
        *scale = abs_max / qmax;
        return HIPQ_SUCCESS;
    }
    case HIPQ_PARAMS_AFFINE: {
        if (!finite || mn > mx) return HIPQ_INVALID_ARGUMENT;
        if (fabsf(mx - mn) < FLT_EPSILON) {
            *zp = qmin_i;
            return HIPQ_SUCCESS;
        }
        float s = (mx - mn) / (qmax - qmin);
        float z = qmin - mn / s;
        *scale = s;
        *zp = f32_as_i32(clamp_keep_nan(roundf(z), qmin, qmax));
        return HIPQ_SUCCESS;
    }
    case HIPQ_PARAMS_BACKEND_SYMMETRIC: {
        if (!finite || mn > mx) return HIPQ_INVALID_ARGUMENT;
        float r = fmaxf(fabsf(mx), fabsf(mn));
        if (r != 0.0f) *scale = (2.0f * r) / (qmax - qmin);
        return HIPQ_SUCCESS;
    }
    case HIPQ_PARAMS_BACKEND_ASYMMETRIC: {
        if (!finite || mn > mx) return HIPQ_INVALID_ARGUMENT;
        if (mx == mn) {
            *zp = qmin_i;
            return HIPQ_SUCCESS;
        }
        float s = (mx - mn) / (qmax - qmin);
        float z = qmin - mn / s;
        *scale = s;
        *zp = f32_as_i32(clamp_keep_nan(roundf(z), qmin, qmax));
        return HIPQ_SUCCESS;
    }
    case HIPQ_PARAMS_ZERO_INCLUDED: {
        mn = fminf(mn, 0.0f);
        mx = fmaxf(mx, 0.0f);
        if (!((fabsf(mn) <= FLT_MAX) && (fabsf(mx) <= FLT_MAX))) return HIPQ_INVALID_ARGUMENT;
        float s = (mx - mn) / (qmax - qmin);
        if (s == 0.0f) s = 1.0f;
        *scale = s;
        *zp = f32_as_i32(fminf(fmaxf(roundf(qmin - mn / s), qmin), qmax));
        return HIPQ_SUCCESS;
    }
    case HIPQ_PARAMS_NN_SYMMETRIC: {
        *scale = fmaxf(fabsf(mx), fabsf(mn)) / 127.0f;
        return HIPQ_SUCCESS;
    }
    case HIPQ_PARAMS_NN_ASYMMETRIC: {
        const float s = (mx - mn) / 255.0f;
        *scale = s;
        *zp = f32_as_i32(roundf(-mn / s));
        return HIPQ_SUCCESS;
    }
    default:
        return HIPQ_INVALID_ARGUMENT;
    }
}

}  // namespace hipq
