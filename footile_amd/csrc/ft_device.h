// ft_device.h -- device-side arithmetic shared by the gfx950 kernels.
//
// 16.16 fixed point with the release-build semantics of footile's Fixed
// (src/fixed.rs): i32 add/sub wrap, mul/div go through i64 and truncate back,
// f32 -> Fixed truncates toward zero with saturation (NaN -> 0).
#pragma once

#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define FT_HD __host__ __device__
#else
#define FT_HD
#endif
#define FT_INLINE FT_HD inline __attribute__((always_inline))

namespace ft {

constexpr int32_t FX_ONE = 65536;
constexpr int32_t FX_HALF = 32768;
constexpr int32_t FX_MASK = 0xFFFF;

FT_HD inline int32_t wadd(int32_t a, int32_t b) { return (int32_t)((uint32_t)a + (uint32_t)b); }
FT_HD inline int32_t wsub(int32_t a, int32_t b) { return (int32_t)((uint32_t)a - (uint32_t)b); }

// Fixed * Fixed, src/fixed.rs:40-47
FT_HD inline int32_t fx_mul(int32_t a, int32_t b) {
    return (int32_t)(uint32_t)(uint64_t)(((int64_t)a * (int64_t)b) >> 16);
}
// 24-bit multiplies: full rate on gfx950, where 32-bit ones (and the 64-bit
// multiply-adds that fx_mul needs) take four times as long.
FT_HD inline uint32_t mul24_u(uint32_t a, uint32_t b) {  // low 32 bits; a, b < 2^24
#if defined(__HIP_DEVICE_COMPILE__)
    return __umul24(a, b);
#else
    return a * b;
#endif
}
FT_HD inline int32_t mul24_i(int32_t a, int32_t b) {  // low 32 bits; -2^23 <= a, b < 2^23
#if defined(__HIP_DEVICE_COMPILE__)
    return __mul24(a, b);
#else
    return (int32_t)((uint32_t)a * (uint32_t)b);
#endif
}
// fx_mul of a, b in [0, ONE] (the product of 65535 and ONE is the largest in 32 bits).
FT_HD inline int32_t fx_mul_unit(int32_t a, int32_t b) {
    return a < FX_ONE ? (int32_t)(mul24_u((uint32_t)a, (uint32_t)b) >> 16) : b;
}
// fx_mul of any a and b in [0, ONE]: a = 2^16 h + l, so a b / 2^16 is h b plus
// l b / 2^16, exactly (the second is the only part with a fraction), mod 2^32.
FT_HD inline int32_t fx_mul_frac(int32_t a, int32_t b) {
    const uint32_t l = mul24_u((uint32_t)a & 0xFFFFu, (uint32_t)b);  // at most 65535 * 65536
    return (int32_t)((uint32_t)mul24_i(a >> 16, b) + (l >> 16));
}

// The low 32 bits of trunc(+-n / d), n = |a| 2^16 <= 2^47 and 1 <= d <= 2^31
// whole numbers, from an r within 2^-49 of 1 / d relatively: floor(n r) is the
// quotient or one off (its error is below 2^47 2^-49 + 2^-6), and the
// remainder, exact in one fma, tells which.
FT_HD inline int32_t fx_div_from(double n, double d, double r, bool neg) {
    double q = floor(n * r);
    const double m = fma(-q, d, n);
    q += m >= d ? 1.0 : (m < 0.0 ? -1.0 : 0.0);
    const double hi = floor(q * 0x1p-32);
    const uint32_t lo = (uint32_t)fma(-hi, 0x1p32, q);
    return (int32_t)(neg ? 0u - lo : lo);
}

// Fixed / Fixed, src/fixed.rs:49-56 (callers never divide by zero).  On the
// device in doubles: the 64-bit integer division is about 130 instructions,
// 30 of them slow multiplies (k_edges of 13.4 M points: 193 -> 164 us).
FT_HD inline int32_t fx_div(int32_t a, int32_t b) {
#if defined(__HIP_DEVICE_COMPILE__)
    const double n = fabs((double)a) * 65536.0, d = fabs((double)b);
    double r = __builtin_amdgcn_rcp(d);  // good to 2^-24 or better: two Newton steps
    r = fma(fma(-d, r, 1.0), r, r);
    r = fma(fma(-d, r, 1.0), r, r);
    return fx_div_from(n, d, r, (a < 0) != (b < 0));
#else
    return (int32_t)(uint32_t)(uint64_t)(((int64_t)a * 65536) / (int64_t)b);
#endif
}
FT_HD inline int32_t fx_abs(int32_t a) { return a < 0 ? (int32_t)(0u - (uint32_t)a) : a; }
FT_HD inline int32_t fx_floor(int32_t a) { return (int32_t)((uint32_t)a & 0xFFFF0000u); }
FT_HD inline int32_t fx_ceil(int32_t a) { return fx_floor(wadd(a, FX_ONE - 1)); }
FT_HD inline int32_t fx_round(int32_t a) { return fx_floor(wadd(a, FX_HALF)); }
FT_HD inline int32_t fx_fract(int32_t a) { return a & FX_MASK; }
FT_HD inline int32_t fx_avg(int32_t a, int32_t b) { return wadd(a, b) >> 1; }
FT_HD inline int32_t fx_int(int32_t a) { return a >> 16; }  // row_of / min_pix

// `(f * 65536.0) as i32`, src/fixed.rs:88-93
FT_HD inline int32_t fx_from_f32(float f) {
    float v = f * 65536.0f;
    if (v != v) return 0;
    if (v >= 2147483648.0f) return INT32_MAX;
    if (v < -2147483648.0f) return INT32_MIN;
    return (int32_t)v;
}

// pixel_cov, src/fig.rs:677-682: round(fcov << 8) as 0..=256
FT_HD inline int32_t pixel_cov(int32_t fcov) {
    return (int32_t)(int16_t)(fx_round((int32_t)((uint32_t)fcov << 8)) >> 16);
}

// FxPt::widdershins, src/fig.rs:116-119
FT_HD inline bool widdershins(int32_t ax, int32_t ay, int32_t bx, int32_t by) {
    return fx_mul(ax, by) > fx_mul(bx, ay);
}

// pix 0.14 Ch8 multiply: both operands widened to 12 bits, product >> 16.
FT_HD inline uint32_t ch8_widen(uint32_t v) { return (v << 4) | (v >> 4); }
FT_HD inline uint32_t ch8_mul_w(uint32_t lw, uint32_t rw) { return (lw * rw) >> 16; }
FT_HD inline uint32_t sat_add_u8(uint32_t a, uint32_t b) {
    uint32_t s = a + b;
    return s > 255u ? 255u : s;
}

// Map a running signed-area sum (taken mod 2^16 as i16) to coverage 0..255,
// src/fig.rs:629-671 and src/imgbuf.rs:54-66,157-167.
FT_HD inline uint32_t coverage_non_zero(int32_t sum) {
    int32_t s = (int32_t)(int16_t)(uint16_t)(uint32_t)sum;
    return s < 0 ? 0u : (s > 255 ? 255u : (uint32_t)s);
}
FT_HD inline uint32_t coverage_even_odd(int32_t sum) {
    int32_t s = (int32_t)(int16_t)(uint16_t)(uint32_t)sum;
    int32_t v = s & 0xFF;
    int32_t odd = s & 0x100;
    int32_t c = v - odd;  // -256..255: no i16 wrap
    c = c < 0 ? -c : c;
    return c > 255 ? 255u : (uint32_t)c;
}

}  // namespace ft
