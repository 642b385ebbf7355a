/* The one-multiply-add requantize of the convolution kernels (RequantFast in hipq_math.h) against the exact chain
 * clamp(round(fl(fl(fl(acc) * sc) + bias) / s) + zp): wherever its test accepts a value the code has to be the same, for
 * both roundings.  Scales, biases and zero points at random over their range, accumulators at random, near every tie and
 * at the ends of the code range.  And the quotients of FastDiv against /.  Exit status 1 on any mismatch. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>

static uint64_t next(uint64_t *s) {
    *s ^= *s << 13;
    *s ^= *s >> 7;
    *s ^= *s << 17;
    return *s;
}
static float uniform(uint64_t *s) { return (float)(next(s) >> 40) * 0x1p-24f; }

static int clamp_code(float r, int zp) {
    const float v = r + (float)zp;
    return v < -128.0f ? -128 : (v > 127.0f ? 127 : (int)v);
}

int main(void) {
    unsigned long long bad = 0, taken = 0, bad_div = 0;
#pragma omp parallel for reduction(+ : bad, taken) schedule(dynamic)
    for (int job = 0; job < 4000; ++job) {
        uint64_t s = 0x9e3779b97f4a7c15ull * (uint64_t)(job + 1);
        const float scale = job % 4 == 0 ? ldexpf(1.0f, (int)(next(&s) % 12) - 12) : exp2f(-18.0f + 20.0f * uniform(&s));
        const float out = job % 4 == 0 ? ldexpf(1.0f, (int)(next(&s) % 8) - 4) : exp2f(-12.0f + 18.0f * uniform(&s));
        const int zp = job % 5 == 0 ? (int)(next(&s) % 64001) - 32000 : (int)(next(&s) % 256) - 128;
        const float bias = job % 3 == 0 ? -0.0f : (uniform(&s) - 0.5f) * out * exp2f(14.0f * uniform(&s) - 2.0f);
        const float inv = 1.0f / out;
        /* RequantFast */
        const float t = 129.0f + fabsf((float)zp), bq = bias * inv;
        const float eps = (6.0f * t + 6.0f * fabsf(bq) + 4.0f) * 0x1.02p-24f;
        const float a = scale * inv, b = bq + (0.5f + eps), limit = 2.0f * eps;
        for (int i = 0; i < 20000; ++i) {
            /* the accumulator whose quotient is nearest to a tie inside or just outside the code range, or any */
            const double q = (double)((int)(next(&s) % 270) - 135 - zp) + 0.5 * (double)(next(&s) % 2);
            double near = (q * out - bias) / scale + (double)((int)(next(&s) % 5) - 2);
            if (i % 4 == 0) near = (double)(int32_t)next(&s);
            if (!(fabs(near) < 2147483647.0)) continue;
            const int32_t acc = (int32_t)near;
            const float f = fmaf((float)acc, a, b);
            const float fract = f - floorf(f);
            if (!(fract >= limit)) continue; /* left to the exact chain */
            ++taken;
            const float fl = floorf(f);
            const long long code = (fl < -1e9f ? -1000000000LL : (fl > 1e9f ? 1000000000LL : (long long)fl)) + zp;
            const int got = code < -128 ? -128 : (code > 127 ? 127 : (int)code);
            volatile float prod = (float)acc * scale;
            volatile float sum = prod + bias;
            const float quot = sum / out;
            if (got != clamp_code(roundf(quot), zp) || got != clamp_code(rintf(quot), zp)) {
                if (bad < 5) printf("mismatch acc=%d scale=%a bias=%a out=%a zp=%d\n", acc, scale, bias, out, zp);
                ++bad;
            }
        }
    }
#pragma omp parallel for reduction(+ : bad_div) schedule(dynamic)
    for (int job = 0; job < 4000; ++job) {
        uint64_t s = 0xd1b54a32d192ed03ull * (uint64_t)(job + 1);
        const uint32_t d = job < 2000 ? (uint32_t)job + 1 : (uint32_t)(next(&s) % 0x7fffffffu >> (next(&s) % 28)) + 1;
        uint32_t m = 0;
        int shift = 0;
        if (d > 1) { /* FastDiv::by */
            int l = 0;
            while ((1ull << l) < d) ++l;
            m = (uint32_t)((1ull << (31 + l)) / d + 1);
            shift = l - 1;
        }
        for (int i = 0; i < 4000; ++i) {
            const uint32_t k = (uint32_t)(next(&s) % (0x7fffffffu / d + 1));
            const uint32_t n = i < 2 ? (i ? 0x7fffffffu : 0) : (i % 3 ? (uint32_t)(next(&s) >> 33) : k * d + (i % 2 ? 0 : d - 1));
            if (n > 0x7fffffffu) continue;
            const uint32_t q = d == 1 ? n : (uint32_t)(((uint64_t)n * m) >> 32) >> shift;
            if (q != n / d) {
                if (bad_div < 5) printf("mismatch %u / %u = %u\n", n, d, q);
                ++bad_div;
            }
        }
    }
    printf("%llu requantize mismatches over %llu values, %llu of the division\n", bad, taken, bad_div);
    return bad != 0 || bad_div != 0 || taken < 10000000ull;
}
