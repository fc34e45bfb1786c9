// Fp inversion by a binary GCD on 28-bit approximations (the "optimized
// binary GCD" of T. Pornin, 2020, eprint 2020/972), for values in 14 x 28-bit
// limbs.  Fermat's p - 2 power needs ~570 dependent multiplications; this
// runs outer iterations of ~1,300 integer instructions each until every lane
// of the wave is done: 19 to 21 for almost every value, at most 30.  Within an
// iteration there are no data-dependent branches.
//
// Invariants (a, b >= 0, u and v signed, all mod p):  a = u*y,  b = v*y.
// Start a = y, b = p, u = 1, v = 0.  Each outer iteration
//  - approximates a and b by their low 28 bits and their top 30 bits,
//  - runs 28 binary-GCD steps on the approximations (if a is odd: swap when
//    a < b, then a -= b; then a /= 2), recording the update as a matrix
//    [[f0, g0], [f1, g1]] with |f| + |g| <= 2^28,
//  - applies it exactly: a <- (a f0 + b g0) / 2^28, b <- (a f1 + b g1) / 2^28
//    (the low 28 bits are exact, so the divisions are exact), negating a row
//    when its result is negative,
//  - and u <- (u f0 + v g0) / 2^28 mod p, v likewise, the division by 2^28
//    done Montgomery-style (add q p with q = -w p^-1 mod 2^28).
// 28 outer iterations reach a = 0, b = gcd = 1 for every y (2 * 381 - 1 binary
// steps suffice), and one after a = 0 would leave v as it is.  Then v = y^-1 mod p, held as a
// signed value of magnitude below 31p (u and v grow by less than p per
// iteration and are never reduced).
//
// Signed multi-limb values: limbs 0..12 in [0, 2^28), limb 13 signed.
// This header is plain C++ apart from the function qualifier, so the host
// test in tests/c can compile it with g++.
#pragma once

#include <cstdint>

#include "constants.h"

#ifndef VKZG_HD
#define VKZG_HD __host__ __device__ inline
#endif

namespace vkzg_amd {
namespace bgcd {

constexpr int kLimbs = 14;
constexpr uint32_t kMask = (1u << 28) - 1u;
constexpr int kOuter = 30;

// acc += x * y as one v_mad_i64_i32.  A limb the compiler knows to be non-negative
// it multiplies unsigned and corrects for the factor's sign in three more
// instructions; hidden limbs (no instructions) stay signed.
VKZG_HD void mac(int64_t &acc, int32_t x, int32_t y) { acc += (int64_t)x * y; }
VKZG_HD int32_t hidden(int32_t x) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+v"(x));
#endif
    return x;
}

// r = (x f + y g) / 2^28 for non-negative x, y < 2^382 (exact division);
// returns true when the result is negative.
VKZG_HD bool lin_shift(uint32_t (&r)[kLimbs], const int32_t (&x)[kLimbs], const int32_t (&y)[kLimbs],
                       int32_t f, int32_t g) {
    int64_t c = 0;
    mac(c, x[0], f);
    mac(c, y[0], g);
    c >>= 28;  // the low 28 bits are zero
    for (int i = 1; i < kLimbs; i++) {
        mac(c, x[i], f);
        mac(c, y[i], g);
        r[i - 1] = (uint32_t)c & kMask;
        c >>= 28;
    }
    r[kLimbs - 1] = (uint32_t)(int32_t)c;  // signed top limb
    return c < 0;
}

// r = -r for a value with a signed top limb; the result is non-negative.
VKZG_HD void negate(uint32_t (&r)[kLimbs]) {
    int32_t c = 0;
    for (int i = 0; i < kLimbs - 1; i++) {
        c -= (int32_t)r[i];
        r[i] = (uint32_t)c & kMask;
        c >>= 28;
    }
    r[kLimbs - 1] = (uint32_t)(c - (int32_t)r[kLimbs - 1]);
}

// r = (u f + v g + q p) / 2^28 with q = -(u f + v g) p^-1 mod 2^28, for signed
// u, v (limbs 0..12 unsigned, limb 13 signed).
VKZG_HD void lin_shift_mod(int32_t (&r)[kLimbs], const int32_t (&u)[kLimbs], const int32_t (&v)[kLimbs],
                           int32_t f, int32_t g) {
    int64_t c = 0;
    mac(c, u[0], f);
    mac(c, v[0], g);
    const int32_t q = hidden((int32_t)(((uint32_t)c * cfp::GCD_N0) & kMask));
    mac(c, q, (int32_t)cfp::GCD_P[0]);
    c >>= 28;
    for (int i = 1; i < kLimbs; i++) {
        mac(c, u[i], f);
        mac(c, v[i], g);
        mac(c, q, (int32_t)cfp::GCD_P[i]);
        r[i - 1] = (int32_t)((uint32_t)c & kMask);
        c >>= 28;
    }
    r[kLimbs - 1] = (int32_t)c;
}

// Low 28 bits and bits [s, s + 30) of x, as a 58-bit approximation.
VKZG_HD uint64_t approx(const uint32_t (&x)[kLimbs], int li, int sh) {
    uint32_t x0 = 0, x1 = 0, x2 = 0;
    for (int i = 0; i < kLimbs; i++) {
        const bool at = i == li;
        x0 = at ? x[i] : x0;
        x1 = at ? (i + 1 < kLimbs ? x[i + 1] : 0u) : x1;
        x2 = at ? (i + 2 < kLimbs ? x[i + 2] : 0u) : x2;
    }
    uint32_t top = x0 >> sh;
    top |= x1 << (28 - sh);
    if (sh > 26) top |= x2 << (56 - sh);
    top &= (1u << 30) - 1u;
    return (uint64_t)(x[0] & kMask) | ((uint64_t)top << 28);
}

// v = y^-1 mod p (signed, |v| < 31p) for y in [1, 2^382) with y != 0 mod p.
// Returns false if the iteration bound was not enough (never observed).
VKZG_HD bool inverse(int32_t (&v)[kLimbs], const uint32_t (&y)[kLimbs]) {
    uint32_t a[kLimbs], b[kLimbs];
    int32_t u[kLimbs];
    for (int i = 0; i < kLimbs; i++) {
        a[i] = y[i];
        b[i] = cfp::GCD_P[i];
        u[i] = 0;
        v[i] = 0;
    }
    u[0] = 1;
    for (int it = 0; it < kOuter; it++) {
        // n = max(len(a), len(b), 58); approximation window s = n - 30
        int hi = 0;
        uint32_t topv = 0;
        for (int i = 0; i < kLimbs; i++) {
            const uint32_t t = a[i] | b[i];
            if (t) {
                hi = i;
                topv = t;
            }
        }
        int len = 28 * hi + (topv ? 32 - __builtin_clz(topv) : 0);
        if (len < 58) len = 58;
        const int s = len - 30;
        const int li = s / 28, sh = s - 28 * li;
        uint64_t ah = approx(a, li, sh), bh = approx(b, li, sh);
        // two runs of 14 steps, each with its rows as one word f + 2^16 g (every
        // step is linear in them, and |f|, |g| <= 2^14 after 14 steps)
        int32_t f0 = 1, g0 = 0, f1 = 0, g1 = 1;
        for (int half = 0; half < 2; half++) {
            int32_t r0 = 1, r1 = 1 << 16;
            for (int j = 0; j < 14; j++) {
                // a odd: a - b; negative: b takes a, and a the difference's
                // magnitude (the swap).  Masks instead of selects: a comparison's
                // lane mask would go through the scalar unit and back.
                const int64_t odd = -(int64_t)(ah & 1u);
                const int64_t d = (int64_t)(ah - (bh & (uint64_t)odd));
                const int64_t neg = d >> 63;
                bh += (uint64_t)(d & neg);
                ah = (uint64_t)((d ^ neg) - neg) >> 1;
                const int32_t rd = r0 - (r1 & (int32_t)odd);
                r1 = (r1 + (rd & (int32_t)neg)) * 2;
                r0 = (rd ^ (int32_t)neg) - (int32_t)neg;
            }
            const int32_t p0 = (int16_t)r0, p1 = (int16_t)r1;
            const int32_t q0 = (r0 - p0) >> 16, q1 = (r1 - p1) >> 16;
            const int32_t tf0 = f0, tg0 = g0;
            f0 = p0 * tf0 + q0 * f1;
            g0 = p0 * tg0 + q0 * g1;
            f1 = p1 * tf0 + q1 * f1;
            g1 = p1 * tg0 + q1 * g1;
        }
        uint32_t na[kLimbs], nb[kLimbs];
        int32_t xa[kLimbs], xb[kLimbs], xu[kLimbs], xv[kLimbs];
        for (int i = 0; i < kLimbs; i++) {
            xa[i] = hidden((int32_t)a[i]);
            xb[i] = hidden((int32_t)b[i]);
            xu[i] = hidden(u[i]);
            xv[i] = hidden(v[i]);
        }
        if (lin_shift(na, xa, xb, f0, g0)) {
            negate(na);
            f0 = -f0;
            g0 = -g0;
        }
        if (lin_shift(nb, xa, xb, f1, g1)) {
            negate(nb);
            f1 = -f1;
            g1 = -g1;
        }
        int32_t nu[kLimbs], nv[kLimbs];
        lin_shift_mod(nu, xu, xv, f0, g0);
        lin_shift_mod(nv, xu, xv, f1, g1);
        uint32_t left = 0;
        for (int i = 0; i < kLimbs; i++) {
            a[i] = na[i];
            b[i] = nb[i];
            u[i] = nu[i];
            v[i] = nv[i];
            left |= na[i];
        }
        // a = 0: what is left would only multiply v by 2^28 and divide it again
        if (left == 0) break;
    }
    uint32_t bad = b[0] ^ 1u;
    for (int i = 0; i < kLimbs; i++) bad |= a[i] | (i ? b[i] : 0u);
    return bad == 0;
}

}  // namespace bgcd
}  // namespace vkzg_amd
