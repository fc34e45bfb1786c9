// BLS12-381 Fp in registers: 13 signed limbs of 30 bits (one per 32-bit
// word), Montgomery form with radix R = 2^390.
//
// Limbs are balanced: a limb is at most 2^29 in magnitude (2^29 + 8 after the
// carry pass of fp_norm), the top one holds what remains (bits 360 up).
//  - A limb product is then below 2^58, so a Montgomery column (13 products,
//    13 of the reduction, the carry) fits a signed 64-bit accumulator and each
//    product is one v_mad_i64_i32 with no carry handling.  Those multiply-adds
//    are what bounds every point kernel (4.8 cycles each on the MI355X against
//    4.2 for other instructions), and 13 limbs take 338 of them per Montgomery
//    product; the 14 x 28-bit unsigned form before took 392, and 32-bit limbs
//    need a carry instruction with each.
//  - p is 381 bits, so 9 bits of headroom stay in the top limb: a value is any
//    residue within +-32p, sums and differences are limb by limb with no
//    conditional correction by p, and a Montgomery product of values of
//    magnitude A p and B p with A B <= 256 is strictly below p in magnitude
//    (A B p / R + 1/2 + 2^-28 < 0.91).
// Measured at two waves per SIMD against the 14 x 28-bit form, in cycles of a
// wave: mixed addition 22,290 -> 17,570, square 1,900 -> 1,610, product 2,440
// -> 2,370 (the additions around the products cost the old form more than they
// do here, where they are limb by limb or folded into a product's carries).
//
// Two operand classes, by the size of the limbs (the top limb apart, which
// stays below 2^26):
//   N   at most 2^29 + 8: products, constants, fp_add, fp_sub, fp_neg, fp_norm
//   N2  at most twice that: fp_add_raw / fp_sub_raw of two N values, FpU digits
// A product takes N2 x N (or N x N2), a square N, a sum of two products N x N
// twice: with |P[i]| the balanced limbs of p, the worst column of N2 x N is
// below 2^62.92, of N2 x N2 or three N x N it could pass 2^63.
//
// Plain C++ apart from the function qualifier, so tests/c builds it with g++.
#pragma once

#include <cstdint>

#include "constants.h"
#include "inverse.h"

#ifndef VKZG_DEV
#define VKZG_DEV __device__ __forceinline__
#endif

namespace vkzg_amd {

constexpr int kFpLimbs = 13;
constexpr int kFpBits = 30;
constexpr uint32_t kFpMask = (1u << kFpBits) - 1u;

struct Fp {
    int32_t v[kFpLimbs];
};
// An integer in unsigned 30-bit digits (byte encodings, comparisons).
struct FpU {
    uint32_t v[kFpLimbs];
};

VKZG_DEV Fp fp_zero() {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = 0;
    return r;
}
VKZG_DEV Fp fp_const(const int32_t (&c)[kFpLimbs]) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = c[i];
    return r;
}
VKZG_DEV Fp fp_one() { return fp_const(cfp::ONE); }

// The low 30 bits of x as a signed digit in [-2^29, 2^29).
VKZG_DEV int32_t fp_digit(uint32_t x) { return (int32_t)(x << (32 - kFpBits)) >> (32 - kFpBits); }
// acc += x * y, one v_mad_i64_i32.
VKZG_DEV void fp_mac(int64_t &acc, int32_t x, int32_t y) { acc += (int64_t)x * y; }
// Values the compiler may not look through (no instructions).  Hiding the
// carry between two columns keeps it from summing every column from zero and
// adding the carry apart (a mixed addition's loop: 4276 -> 4128 instructions and
// 229 -> 175 VGPRs); a hidden multiplier keeps a folded value one multiply-add
// per limb instead of a sign extension and a 64-bit subtraction (4128 -> 4021,
// 136 VGPRs).
#if defined(__HIP_DEVICE_COMPILE__)
VKZG_DEV void fp_hide(int64_t &acc) { asm("" : "+v"(acc)); }
VKZG_DEV int32_t fp_hidden(int32_t k) {
    asm("" : "+s"(k));
    return k;
}
#else
VKZG_DEV void fp_hide(int64_t &) {}
VKZG_DEV int32_t fp_hidden(int32_t k) { return k; }
#endif

// The Montgomery product by product scanning.  col(acc, i) adds column i of
// the product(s); column k of m*p shares the accumulator, m_k makes the low 30
// bits of columns k < 13 vanish, and the accumulator shifts down one limb per
// column.  fold(acc, i) adds limb i of a value that is added to the result
// (X3 = R^2 - PPP - 2Q and the like): one v_mad_i64_i32 per limb, where a
// separate subtraction would need a carry pass of its own.  Result digits are
// taken with a rounding carry, so they are strictly balanced: a result that is
// 0 mod p is the zero limbs (its magnitude is below p).
template <typename Col, typename Fold>
VKZG_DEV Fp fp_mont(Col col, Fold fold) {
    int32_t m[kFpLimbs];
    int64_t acc = 0;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) {
        col(acc, i);
#pragma unroll
        for (int j = 0; j < i; j++) fp_mac(acc, m[j], cfp::P[i - j]);
        m[i] = fp_digit((uint32_t)acc * cfp::N0);
        fp_mac(acc, m[i], cfp::P[0]);
        acc >>= kFpBits;
        fp_hide(acc);
    }
    Fp r;
#pragma unroll
    for (int i = kFpLimbs; i < 2 * kFpLimbs - 1; i++) {
        col(acc, i);
        fold(acc, i - kFpLimbs);
#pragma unroll
        for (int j = i - kFpLimbs + 1; j < kFpLimbs; j++) fp_mac(acc, m[j], cfp::P[i - j]);
        r.v[i - kFpLimbs] = fp_digit((uint32_t)acc);
        acc = (acc + (1 << (kFpBits - 1))) >> kFpBits;
        fp_hide(acc);
    }
    fold(acc, kFpLimbs - 1);
    r.v[kFpLimbs - 1] = (int32_t)acc;
    return r;
}

// Column i of a * b, and of a^2 from a and 2a (91 limb products instead of 169).
VKZG_DEV void fp_col(int64_t &acc, int i, const Fp &a, const Fp &b) {
#pragma unroll
    for (int j = 0; j < kFpLimbs; j++)
        if (i - j >= 0 && i - j < kFpLimbs) fp_mac(acc, a.v[j], b.v[i - j]);
}
VKZG_DEV void fp_col_sqr(int64_t &acc, int i, const Fp &a, const Fp &a2) {
#pragma unroll
    for (int j = 0; j < kFpLimbs; j++) {
        if (2 * j < i && i - j < kFpLimbs) fp_mac(acc, a2.v[j], a.v[i - j]);
        if (2 * j == i) fp_mac(acc, a.v[j], a.v[j]);
    }
}

// Limb by limb, N inputs to an N2 result.
VKZG_DEV Fp fp_add_raw(const Fp &a, const Fp &b) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = a.v[i] + b.v[i];
    return r;
}
VKZG_DEV Fp fp_sub_raw(const Fp &a, const Fp &b) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = a.v[i] - b.v[i];
    return r;
}
VKZG_DEV Fp fp_dbl_raw(const Fp &a) { return fp_add_raw(a, a); }

VKZG_DEV Fp fp_mul(const Fp &a, const Fp &b) {
    return fp_mont([&](int64_t &acc, int i) { fp_col(acc, i, a, b); }, [](int64_t &, int) {});
}
VKZG_DEV Fp fp_sqr(const Fp &a) {
    const Fp a2 = fp_dbl_raw(a);
    return fp_mont([&](int64_t &acc, int i) { fp_col_sqr(acc, i, a, a2); }, [](int64_t &, int) {});
}
// a b + k c, a^2 + k c and a^2 + k c + l d with the added values' limbs any
// 32-bit ones and |k|, |l| <= 8 (fp_mul_fold_v: k may differ from lane to
// lane).  The result is balanced; its magnitude is that of the product (below
// p) plus those of the added values.
VKZG_DEV Fp fp_mul_fold_v(const Fp &a, const Fp &b, const Fp &c, int32_t k) {
    return fp_mont([&](int64_t &acc, int i) { fp_col(acc, i, a, b); },
                   [&](int64_t &acc, int i) { fp_mac(acc, c.v[i], k); });
}
VKZG_DEV Fp fp_mul_fold(const Fp &a, const Fp &b, const Fp &c, int32_t k) {
    return fp_mul_fold_v(a, b, c, fp_hidden(k));
}
VKZG_DEV Fp fp_sqr_fold(const Fp &a, const Fp &c, int32_t k) {
    const Fp a2 = fp_dbl_raw(a);
    k = fp_hidden(k);
    return fp_mont([&](int64_t &acc, int i) { fp_col_sqr(acc, i, a, a2); },
                   [&](int64_t &acc, int i) { fp_mac(acc, c.v[i], k); });
}
VKZG_DEV Fp fp_sqr_fold2(const Fp &a, const Fp &c, int32_t k, const Fp &d, int32_t l) {
    const Fp a2 = fp_dbl_raw(a);
    k = fp_hidden(k);
    l = fp_hidden(l);
    return fp_mont([&](int64_t &acc, int i) { fp_col_sqr(acc, i, a, a2); },
                   [&](int64_t &acc, int i) {
                       fp_mac(acc, c.v[i], k);
                       fp_mac(acc, d.v[i], l);
                   });
}
// a b + c d under one reduction (507 limb products instead of 676), all N.
VKZG_DEV Fp fp_mul_sum(const Fp &a, const Fp &b, const Fp &c, const Fp &d) {
    return fp_mont(
        [&](int64_t &acc, int i) {
            fp_col(acc, i, a, b);
            fp_col(acc, i, c, d);
        },
        [](int64_t &, int) {});
}

// One carry pass, every limb's carry at once (no chain): limbs of magnitude
// below 3 * 2^29 (the sum of two N values, three times a product) come back as
// N.
VKZG_DEV Fp fp_norm(const Fp &a) {
    Fp r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < kFpLimbs - 1; i++) {
        r.v[i] = fp_digit((uint32_t)a.v[i]) + c;
        c = (a.v[i] + (1 << (kFpBits - 1))) >> kFpBits;
    }
    r.v[kFpLimbs - 1] = a.v[kFpLimbs - 1] + c;
    return r;
}
// The same for any 32-bit limbs.
VKZG_DEV Fp fp_norm_wide(const Fp &a) {
    Fp r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < kFpLimbs - 1; i++) {
        r.v[i] = fp_digit((uint32_t)a.v[i]) + c;
        c = ((a.v[i] >> (kFpBits - 1)) + 1) >> 1;
    }
    r.v[kFpLimbs - 1] = a.v[kFpLimbs - 1] + c;
    return r;
}
VKZG_DEV Fp fp_add(const Fp &a, const Fp &b) { return fp_norm(fp_add_raw(a, b)); }
VKZG_DEV Fp fp_sub(const Fp &a, const Fp &b) { return fp_norm(fp_sub_raw(a, b)); }
VKZG_DEV Fp fp_dbl(const Fp &a) { return fp_norm(fp_dbl_raw(a)); }
// 3a of a product (strictly balanced digits)
VKZG_DEV Fp fp_triple(const Fp &a) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = 3 * a.v[i];
    return fp_norm(r);
}
// 2a - b
VKZG_DEV Fp fp_dbl_sub(const Fp &a, const Fp &b) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = 2 * a.v[i] - b.v[i];
    return fp_norm_wide(r);
}
VKZG_DEV Fp fp_neg(const Fp &a) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = -a.v[i];
    return r;
}
// neg ? -a : a, as (a ^ s) - s with s = 0 or -1
VKZG_DEV Fp fp_cond_neg(const Fp &a, bool neg) {
    const int32_t s = neg ? -1 : 0;
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = (a.v[i] ^ s) - s;
    return r;
}
// c ? a : b limb by limb (v_cndmask), so a lane-varying choice between two
// register values never goes through an address.
VKZG_DEV Fp fp_select(bool c, const Fp &a, const Fp &b) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = c ? a.v[i] : b.v[i];
    return r;
}
// The value of lane q of a quad: a, b, c or d.
VKZG_DEV Fp fp_select4(uint32_t q, const Fp &a, const Fp &b, const Fp &c, const Fp &d) {
    return fp_select((q & 2u) != 0, fp_select((q & 1u) != 0, d, c), fp_select((q & 1u) != 0, b, a));
}

// Zero mod p, for a value whose residue 0 has one form only: a product, a
// constant, or a small multiple or negation of one (magnitude of the product
// below p, digits balanced).
VKZG_DEV bool fp_is_zero(const Fp &a) {
    int32_t z = 0;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) z |= a.v[i];
    return z == 0;
}
// The same residue with magnitude below p, for any N2 value of magnitude up to
// 256p (a product by one).  Sums have no other correction, so a recurrence
// that adds its own last value without a product between (x <- s - 2x) needs it.
VKZG_DEV Fp fp_reduce(const Fp &a) { return fp_mul(a, fp_one()); }
// Zero mod p for any such value.
VKZG_DEV bool fp_is_zero_mod(const Fp &a) { return fp_is_zero(fp_reduce(a)); }
// a == b mod p, for N values of magnitude up to 128p.
VKZG_DEV bool fp_eq(const Fp &a, const Fp &b) { return fp_is_zero_mod(fp_sub_raw(a, b)); }

// The digits in [0, p) of a value of magnitude below p (a product).
VKZG_DEV FpU fp_canonical(const Fp &a) {
    FpU s, t;
    int32_t cs = 0, ct = 0;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) {
        const int32_t x = a.v[i] + cs;
        s.v[i] = (uint32_t)x & kFpMask;
        cs = x >> kFpBits;
        const int32_t y = (int32_t)s.v[i] + (int32_t)cfp::PU[i] + ct;
        t.v[i] = (uint32_t)y & kFpMask;
        ct = y >> kFpBits;
    }
    FpU r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = cs < 0 ? t.v[i] : s.v[i];
    return r;
}
// Digits as limbs: an N2 operand.
VKZG_DEV Fp fp_from_digits(const FpU &a) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = (int32_t)a.v[i];
    return r;
}
// Montgomery -> canonical integer in [0, p).
VKZG_DEV FpU fp_to_canonical(const Fp &a) {
    Fp one = fp_zero();
    one.v[0] = 1;
    return fp_canonical(fp_mul(a, one));
}
// Integer below 2^390 -> Montgomery form.
VKZG_DEV Fp fp_from_canonical(const FpU &a) { return fp_mul(fp_from_digits(a), fp_const(cfp::R2)); }

// NA digits of BA bits -> NB digits of BB bits of the same integer (bits the
// source does not have read as zero, digits past the target's last are dropped).
template <int BA, int NA, int BB, int NB>
VKZG_DEV void fp_repack(uint32_t (&out)[NB], const uint32_t (&in)[NA]) {
    constexpr uint32_t mask = BB == 32 ? 0xffffffffu : (1u << (BB & 31)) - 1u;
#pragma unroll
    for (int k = 0; k < NB; k++) {
        const int bit = BB * k, li = bit / BA, sh = bit % BA;
        uint32_t x = li < NA ? in[li] >> sh : 0u;
        if (BA - sh < BB && li + 1 < NA) x |= in[li + 1] << (BA - sh);
        if (2 * BA - sh < BB && li + 2 < NA) x |= in[li + 2] << (2 * BA - sh);
        out[k] = x & mask;
    }
}
// 12 little-endian 32-bit words (a value below 2^384) <-> digits.
VKZG_DEV FpU fp_from_words(const uint32_t (&w)[12]) {
    FpU r;
    fp_repack<32, 12, kFpBits, kFpLimbs>(r.v, w);
    return r;
}
VKZG_DEV void fp_to_words(uint32_t (&w)[12], const FpU &a) { fp_repack<kFpBits, kFpLimbs, 32, 12>(w, a.v); }
// a < m in digits
VKZG_DEV bool fp_digits_lt(const FpU &a, const uint32_t (&m)[kFpLimbs]) {
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) c = ((int32_t)a.v[i] - (int32_t)m[i] + c) >> kFpBits;
    return c < 0;
}
VKZG_DEV bool fp_limbs_lt_p(const FpU &a) { return fp_digits_lt(a, cfp::PU); }
// canonical value > (p-1)/2 (the sign flag of the compressed encoding)
VKZG_DEV bool fp_is_lex_largest(const FpU &canonical) {
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++)
        c = ((int32_t)cfp::HALFU[i] - (int32_t)canonical.v[i] + c) >> kFpBits;
    return c < 0;
}
VKZG_DEV bool fpu_is_zero(const FpU &a) {
    uint32_t z = 0;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) z |= a.v[i];
    return z == 0;
}
VKZG_DEV bool fpu_eq(const FpU &a, const FpU &b) {
    uint32_t z = 0;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) z |= a.v[i] ^ b.v[i];
    return z == 0;
}

template <int NE>
VKZG_DEV Fp fp_pow_const(const Fp &a, const uint32_t (&e)[NE]) {
    Fp acc = fp_one();
#pragma unroll 1
    for (int i = NE - 1; i >= 0; i--) {
        const uint32_t limb = e[i];
#pragma unroll 1
        for (int b = 31; b >= 0; b--) {
            acc = fp_sqr(acc);
            if ((limb >> b) & 1u) acc = fp_mul(acc, a);
        }
    }
    return acc;
}
VKZG_DEV Fp fp_inv_fermat(const Fp &a) { return fp_pow_const<12>(a, cfp::P_MINUS_2); }

// a^e for a constant exponent by a sliding window of 4 bits over the odd
// powers a, a^3, ..., a^15: the same squarings as fp_pow_const and about a
// fifth of its multiplications.
template <int NE>
VKZG_DEV Fp fp_pow_const_window(const Fp &a, const uint32_t (&e)[NE]) {
    Fp odd[8];
    odd[0] = a;
    const Fp a2 = fp_sqr(a);
#pragma unroll
    for (int k = 1; k < 8; k++) odd[k] = fp_mul(odd[k - 1], a2);
    Fp acc = fp_one();
    int i = NE * 32 - 1;
    while (i >= 0 && !((e[i / 32] >> (i % 32)) & 1u)) i--;
    bool started = false;
#pragma unroll 1
    while (i >= 0) {
        if (!((e[i / 32] >> (i % 32)) & 1u)) {
            acc = fp_sqr(acc);
            i--;
            continue;
        }
        // longest window of at most 4 bits ending in a set bit
        int j = i - 3 < 0 ? 0 : i - 3;
        while (!((e[j / 32] >> (j % 32)) & 1u)) j++;
        uint32_t w = 0;
        for (int k = i; k >= j; k--) w = (w << 1) | ((e[k / 32] >> (k % 32)) & 1u);
        if (started) {
            for (int k = i; k >= j; k--) acc = fp_sqr(acc);
            acc = fp_mul(acc, odd[w >> 1]);
        } else {
            acc = odd[w >> 1];
            started = true;
        }
        i = j - 1;
    }
    return acc;
}

// Inverse of a Montgomery value xR (0 -> 0), for any N2 value of magnitude up
// to 256p: its integer in [0, p) goes through the binary GCD of inverse.h (28-bit
// limbs), which gives the plain inverse (xR)^-1 as a signed value in
// (-31p, 31p); adding 32p makes it non-negative and a Montgomery product by
// R^3 turns it into x^-1 R.
VKZG_DEV Fp fp_inv(const Fp &a) {
    const Fp x = fp_reduce(a);
    if (fp_is_zero(x)) return fp_zero();
    const FpU u = fp_canonical(x);
    uint32_t y[bgcd::kLimbs], t[bgcd::kLimbs];
    fp_repack<kFpBits, kFpLimbs, 28, bgcd::kLimbs>(y, u.v);
    int32_t v[bgcd::kLimbs];
    if (!bgcd::inverse(v, y)) return fp_inv_fermat(x);
    int64_t c = 0;
#pragma unroll
    for (int i = 0; i < bgcd::kLimbs; i++) {
        c += (int64_t)v[i] + cfp::GCD_P32[i];
        t[i] = (uint32_t)c & bgcd::kMask;
        c >>= 28;
    }
    FpU w;
    fp_repack<28, bgcd::kLimbs, kFpBits, kFpLimbs>(w.v, t);
    return fp_mul(fp_from_digits(w), fp_const(cfp::R3_M));
}

// Reference Montgomery product (operand scanning) for the test hooks: the
// same radix, canonical.
VKZG_DEV FpU fp_mul_reference(const Fp &a, const Fp &b) {
    int64_t t[kFpLimbs + 1];
#pragma unroll
    for (int j = 0; j <= kFpLimbs; j++) t[j] = 0;
    for (int i = 0; i < kFpLimbs; i++) {
        for (int j = 0; j < kFpLimbs; j++) t[j] += (int64_t)a.v[j] * b.v[i];
        const int32_t m = fp_digit((uint32_t)t[0] * cfp::N0);
        for (int j = 0; j < kFpLimbs; j++) t[j] += (int64_t)m * cfp::P[j];
        t[1] += t[0] >> kFpBits;  // exact: the low 30 bits are zero
        for (int j = 0; j < kFpLimbs; j++) t[j] = t[j + 1];
        t[kFpLimbs] = 0;
    }
    Fp r;
    for (int j = 0; j < kFpLimbs - 1; j++) {
        r.v[j] = fp_digit((uint32_t)t[j]);
        t[j + 1] += (t[j] + (1 << (kFpBits - 1))) >> kFpBits;
    }
    r.v[kFpLimbs - 1] = (int32_t)t[kFpLimbs - 1];
    return fp_canonical(r);
}

}  // namespace vkzg_amd
