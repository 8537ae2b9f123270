// bla_key.hpp -- radii of the BLA table as integer keys, so that a lookup
// compares |z| with a radius without taking a square root.
//
// The reference's test is sqrt(q) < r with q = x^2 + y^2 and a correctly
// rounded square root (on a value scaled by a power of two, which is exact).
// The rounded square root never decreases with q, so for every r = m 2^e
// (m in [1, 2)) there is a least binary64 t with sqrt(t) >= m, and
//     sqrt(q 2^(2 e1)) < m 2^e   if and only if   q 2^(2 e1) < t 2^(2 e).
// A key is the right-hand side as one signed 64-bit integer: the bits of the
// positive binary64 with 2 e added to the exponent field, which is then
// signed and may lie outside the binary64 range.  Keys are ordered as the
// values are, so the test is one integer comparison per radius.  The square
// root it replaces is a sequence of about 20 binary64 instructions on
// gfx950, plus one v_ldexp_f64 per radius read
// (2048x2048 frames: 1e-300 -2 %, 1e-2000 -3 %, interior-dominated -4.6 %).
#pragma once
#include "xr.hpp"

namespace fsg {

// Exponents are clamped to what the field holds: below KEY_MIN_E |z| is under
// every nonzero radius (2^-1074 at least); from 2^KEY_MAX_E on, where |z|^2
// leaves the binary64 range, |z| is under no finite radius.
constexpr int32_t KEY_MIN_E = -1100, KEY_MAX_E = 511;

// key of a radius: nothing is below a zero (or NaN) radius, everything
// finite below an infinite one
FSG_HD int64_t radius_key(double r) {
    if (!(r > 0.)) return INT64_MIN;
    if (r > 1.7976931348623157e308) return INT64_MAX;
    int e;
    const double m = 2. * frexp(r, &e);      // [1, 2), exact for a subnormal r too
    e -= 1;
    if (e >= KEY_MAX_E) return (int64_t)(1023 + 2 * KEY_MAX_E) << 52;
    double t = m * m;
    while (sqrt(t) >= m) t = from_bits(bits(t) - 1);
    while (sqrt(t) < m) t = from_bits(bits(t) + 1);
    return (int64_t)bits(t) + (int64_t)e * ((int64_t)1 << 53);
}

// key of |z|^2 = q 2^(2 e), q >= 1 (a zero q, from a zero z, counts as 1:
// its exponent lies below KEY_MIN_E)
FSG_HD int64_t modulus_key(double q, int32_t e) {
    const uint64_t b = bits(q);
    const int32_t hq = (int32_t)(b >> 32);
    const int32_t ec = min(max(e, KEY_MIN_E), KEY_MAX_E);
    const uint32_t hi = (uint32_t)max(hq, 0x3ff00000) + ((uint32_t)ec << 21);
    return (int64_t)(((uint64_t)hi << 32) | (uint32_t)b);
}

// key of |x + iy| for binary64 x, y, deciding as hypot2(x, y) < r does
FSG_HD int64_t hypot_key(double x, double y) {
    const double mx = fmax(fabs(x), fabs(y));
    // The prescale by a power of two is exact and leaves the key as it is: not
    // needed while the larger square's last place lies above the subnormal
    // range (a smaller square that is subnormal is then below half of it).
    if (mx >= 0x1p-480 && mx <= 0x1p500) return (int64_t)bits(x * x + y * y);
    if (!(mx >= 0x1p-900 && mx <= 0x1p500)) {            // zero, tiny, huge or NaN
        const double h = hypot2(x, y);
        return h == h ? radius_key(h) : INT64_MAX;
    }
    int e;
#ifdef __HIP_DEVICE_COMPILE__
    e = __builtin_amdgcn_frexp_exp(mx) - 1;
#else
    (void)frexp(mx, &e);
    e -= 1;
#endif
    const double xs = ldexp(x, -e), ys = ldexp(y, -e);
    return (int64_t)bits(xs * xs + ys * ys) + (int64_t)((uint64_t)(uint32_t)e << 53);   // in range: no clamp
}

}  // namespace fsg
