// BLS12-381 G1 (y^2 = x^3 + 4) point arithmetic for gfx950.
//
// Three representations:
//   G1A  affine (x, y), with (0, 0) standing for the identity (it is not on
//        the curve), as in the reference (src/shaders/field.glsl.inc:304-320);
//   G1J  Jacobian (X, Y, Z), x = X/Z^2, y = Y/Z^3, Z = 0 is the identity --
//        used for doubling chains (dbl-2009-l, 2M+5S);
//   G1X  extended Jacobian "XYZZ" (X, Y, ZZ, ZZZ), x = X/ZZ, y = Y/ZZZ,
//        ZZ = 0 is the identity -- used for accumulation (madd-2008-s 8M+2S,
//        add-2008-s 12M+2S), cheaper than the reference's Jacobian madd
//        (7M+4S) and add (11M+5S).
// Every addition handles P == Q (falls back to doubling) and P == -Q.
#pragma once

#include "field.h"

// Point additions and doublings are inlined into the kernels (passing 100-200
// byte points to an out-of-line function goes through the stack in scratch
// memory, which measured at several times the kernels' useful HBM traffic).
// The P == Q fallbacks inside additions are rare and stay out of line.
#define VKZG_DEV_CALL __device__ __forceinline__
#define VKZG_DEV_COLD __device__ __forceinline__

namespace vkzg_amd {

struct G1A {
    Fp x, y;
};
struct G1J {
    Fp x, y, z;
};
// A phase-A table entry: an affine point padded to exactly one 128-byte
// line, so each random gather touches one line instead of two.
struct __attribute__((aligned(128))) G1AT {
    G1A p;
};
struct G1X {
    Fp x, y, zz, zzz;
};

VKZG_DEV G1A g1a_identity() {
    G1A r;
    r.x = fp_zero();
    r.y = fp_zero();
    return r;
}
VKZG_DEV bool g1a_is_identity(const G1A &p) { return fp_is_zero(p.x) && fp_is_zero(p.y); }
VKZG_DEV G1A g1a_neg_if(const G1A &p, bool neg) {
    G1A r;
    r.x = p.x;
    // The identity (0, 0) stays (0, 0): fp_neg(0) == 0.
    r.y = fp_cond_neg(p.y, neg);
    return r;
}

// ---------------------------------------------------------------- Jacobian

VKZG_DEV G1J g1j_identity() {
    G1J r;
    r.x = fp_one();
    r.y = fp_one();
    r.z = fp_zero();
    return r;
}
VKZG_DEV G1J g1j_from_affine(const G1A &a) {
    if (g1a_is_identity(a)) return g1j_identity();
    G1J r;
    r.x = a.x;
    r.y = a.y;
    r.z = fp_one();
    return r;
}

// dbl-2009-l with its additions folded into the products: W = 2 X Y^2,
// X3 = E^2 - 4W, Y3 = E (2W - X3) - 8 Y^4, Z3 = 2 Y Z (E = 3 X^2).
VKZG_DEV_CALL G1J g1j_dbl(const G1J &p) {
    if (fp_is_zero(p.z)) return p;
    const Fp E = fp_triple(fp_sqr(p.x));
    const Fp B = fp_sqr(p.y);
    const Fp C = fp_sqr(B);
    const Fp W = fp_mul(fp_dbl_raw(p.x), B);
    G1J r;
    r.x = fp_sqr_fold(E, W, -4);
    r.y = fp_mul_fold(E, fp_dbl_sub(W, r.x), C, -8);
    r.z = fp_mul(fp_dbl_raw(p.y), p.z);
    return r;
}

VKZG_DEV_COLD G1J g1j_dbl_cold(const G1J &p);

// add-2007-bl without its factors of two: H = U2 - U1, R = S2 - S1, V = U1 H^2,
// X3 = R^2 - H^3 - 2V, Y3 = R (V - X3) - S1 H^3, Z3 = Z1 Z2 H.
VKZG_DEV_CALL G1J g1j_add(const G1J &a, const G1J &b) {
    if (fp_is_zero(a.z)) return b;
    if (fp_is_zero(b.z)) return a;
    const Fp Z1Z1 = fp_sqr(a.z);
    const Fp Z2Z2 = fp_sqr(b.z);
    const Fp U1 = fp_mul(a.x, Z2Z2);
    const Fp S1 = fp_mul(a.y, fp_mul(b.z, Z2Z2));
    const Fp H = fp_mul_fold(b.x, Z1Z1, U1, -1);
    const Fp R = fp_mul_fold(b.y, fp_mul(a.z, Z1Z1), S1, -1);
    const Fp HH = fp_sqr(H);
    if (fp_is_zero(HH)) {
        if (fp_is_zero_mod(R)) return g1j_dbl_cold(a);
        return g1j_identity();
    }
    const Fp HHH = fp_mul(H, HH);
    const Fp V = fp_mul(U1, HH);
    G1J r;
    r.x = fp_sqr_fold2(R, HHH, -1, V, -2);
    r.y = fp_mul_sum(R, fp_sub(V, r.x), S1, fp_neg(HHH));
    r.z = fp_mul(fp_mul(a.z, b.z), H);
    return r;
}

VKZG_DEV_COLD G1J g1j_dbl_cold(const G1J &p) { return g1j_dbl(p); }

// The same with b affine and not the identity, a not the identity: H and R
// given, H not 0 mod p.
VKZG_DEV G1J g1j_madd_tail(const G1J &a, const Fp &H, const Fp &HH, const Fp &R) {
    const Fp HHH = fp_mul(H, HH);
    const Fp V = fp_mul(a.x, HH);
    G1J r;
    r.x = fp_sqr_fold2(R, HHH, -1, V, -2);
    r.y = fp_mul_sum(R, fp_sub(V, r.x), a.y, fp_neg(HHH));
    r.z = fp_mul(a.z, H);
    return r;
}

// madd (b affine, may be the identity)
VKZG_DEV_CALL G1J g1j_madd(const G1J &a, const G1A &b) {
    if (g1a_is_identity(b)) return a;
    if (fp_is_zero(a.z)) return g1j_from_affine(b);
    const Fp Z1Z1 = fp_sqr(a.z);
    const Fp H = fp_mul_fold(b.x, Z1Z1, a.x, -1);
    const Fp R = fp_mul_fold(b.y, fp_mul(a.z, Z1Z1), a.y, -1);
    const Fp HH = fp_sqr(H);
    if (fp_is_zero(HH)) {
        if (fp_is_zero_mod(R)) return g1j_dbl_cold(a);
        return g1j_identity();
    }
    return g1j_madd_tail(a, H, HH, R);
}

// Jacobian + affine for hot loops (see g1x_madd_fast for the contract).
VKZG_DEV G1J g1j_madd_fast(const G1J &a, const G1A &b, bool &exc) {
    if (g1a_is_identity(b)) return a;
    if (fp_is_zero(a.z)) return g1j_from_affine(b);
    const Fp Z1Z1 = fp_sqr(a.z);
    const Fp H = fp_mul_fold(b.x, Z1Z1, a.x, -1);
    const Fp R = fp_mul_fold(b.y, fp_mul(a.z, Z1Z1), a.y, -1);
    const Fp HH = fp_sqr(H);
    exc |= fp_is_zero(HH);
    return g1j_madd_tail(a, H, HH, R);
}

VKZG_DEV G1J g1j_neg(const G1J &p) {
    G1J r = p;
    r.y = fp_neg(p.y);
    return r;
}

// ---------------------------------------------------------------- XYZZ

VKZG_DEV G1X g1x_identity() {
    G1X r;
    r.x = fp_one();
    r.y = fp_one();
    r.zz = fp_zero();
    r.zzz = fp_zero();
    return r;
}
VKZG_DEV bool g1x_is_identity(const G1X &p) { return fp_is_zero(p.zz); }
VKZG_DEV G1X g1x_from_affine(const G1A &a) {
    if (g1a_is_identity(a)) return g1x_identity();
    G1X r;
    r.x = a.x;
    r.y = a.y;
    r.zz = fp_one();
    r.zzz = fp_one();
    return r;
}
// (X, Y, ZZ, ZZZ) with ZZ^3 == ZZZ^2 -> Jacobian with Z = ZZ*ZZZ:
// X_J = X*ZZ^4, Y_J = Y*ZZZ^4 (no inversion).
VKZG_DEV_CALL G1J g1j_from_xyzz(const G1X &p) {
    if (fp_is_zero(p.zz)) return g1j_identity();
    G1J r;
    const Fp zz2 = fp_sqr(p.zz);
    const Fp zzz2 = fp_sqr(p.zzz);
    r.x = fp_mul(p.x, fp_sqr(zz2));
    r.y = fp_mul(p.y, fp_sqr(zzz2));
    r.z = fp_mul(p.zz, p.zzz);
    return r;
}

// dbl-2008-s-1 in halves: V = 4 Y^2 and W = 8 Y^3 enter their products as
// twice V2 = 2 Y^2 and W2 = 4 Y^3, so every operand stays within its class.
// The identity (ZZ = ZZZ = 0) doubles to ZZ3 = ZZZ3 = 0, the identity again,
// so no input has to stay live for a select; doubling has no exceptional case.
VKZG_DEV G1X g1x_dbl_core(const G1X &p) {
    const Fp V2 = fp_mul(fp_dbl_raw(p.y), p.y);
    const Fp V = fp_dbl_raw(V2);
    const Fp W2 = fp_mul(V, p.y);
    const Fp S = fp_mul(V, p.x);
    G1X r;
    r.zz = fp_mul(V, p.zz);
    r.zzz = fp_mul(fp_dbl_raw(W2), p.zzz);
    const Fp M = fp_triple(fp_sqr(p.x));
    r.x = fp_sqr_fold(M, S, -2);
    r.y = fp_mul_sum(M, fp_sub(S, r.x), fp_dbl(W2), fp_neg(p.y));
    return r;
}
VKZG_DEV_CALL G1X g1x_dbl(const G1X &p) {
    if (fp_is_zero(p.zz)) return p;
    return g1x_dbl_core(p);
}

VKZG_DEV_COLD G1X g1x_dbl_cold(const G1X &p) { return g1x_dbl(p); }

// The rest of an XYZZ addition once P = U2 - U1, PP = P^2 and R = S2 - S1
// are there: (X1, Y1) are the first point's scaled coordinates (U1, S1; with
// an affine second point its own X and Y), zz and zzz the product of both
// points' ZZ and of both ZZZ.  X3 = R^2 - PPP - 2Q is folded into the square
// and Y3 = R (Q - X3) - Y1 PPP takes one reduction for its two products.
VKZG_DEV G1X g1x_add_tail(const Fp &X1, const Fp &Y1, const Fp &zz, const Fp &zzz, const Fp &P, const Fp &PP,
                          const Fp &R) {
    const Fp PPP = fp_mul(P, PP);
    const Fp Q = fp_mul(X1, PP);
    G1X r;
    r.zz = fp_mul(zz, PP);
    r.zzz = fp_mul(zzz, PPP);
    r.x = fp_sqr_fold2(R, PPP, -1, Q, -2);
    r.y = fp_mul_sum(R, fp_sub(Q, r.x), Y1, fp_neg(PPP));
    return r;
}

// madd-2008-s: XYZZ + affine (b may be the identity)
VKZG_DEV_CALL G1X g1x_madd(const G1X &a, const G1A &b) {
    if (g1a_is_identity(b)) return a;
    if (fp_is_zero(a.zz)) return g1x_from_affine(b);
    const Fp P = fp_mul_fold(b.x, a.zz, a.x, -1);
    const Fp R = fp_mul_fold(b.y, a.zzz, a.y, -1);
    const Fp PP = fp_sqr(P);
    if (fp_is_zero(PP)) {
        if (fp_is_zero_mod(R)) return g1x_dbl_cold(g1x_from_affine(b));
        return g1x_identity();
    }
    return g1x_add_tail(a.x, a.y, a.zz, a.zzz, P, PP, R);
}

// Hot-loop variants.  When the inputs are equal or opposite (the doubling /
// cancellation cases, which random data never reaches) they set `exc` and
// return an unspecified point; callers then recompute that result with the
// checked forms above outside their loops.  Keeping the rare path out of the
// loop body is what keeps the accumulator in VGPRs (a call inside the loop
// that takes the point by address pins it to scratch memory).  P == 0 is
// detected on PP = P^2, whose residue 0 is the zero limbs.

// Accumulator step a + (+-b) for an accumulator that is never the identity
// (callers start it from their first point).  b is an affine point in
// normalised limbs, negated when `neg`; `exc` is also set when b is the
// identity (all-zero limbs: no point of the prime-order group has y = 0).
VKZG_DEV G1X g1x_madd_acc(const G1X &a, const G1A &b, bool neg, bool &exc) {
    exc |= fp_is_zero(b.y);
    const Fp P = fp_mul_fold(b.x, a.zz, a.x, -1);
    const Fp R = fp_mul_fold(fp_cond_neg(b.y, neg), a.zzz, a.y, -1);
    const Fp PP = fp_sqr(P);
    exc |= fp_is_zero(PP);
    return g1x_add_tail(a.x, a.y, a.zz, a.zzz, P, PP, R);
}

// The first point of an accumulator: (+-b) in XYZZ; flags the identity.
VKZG_DEV G1X g1x_start(const G1A &b, bool neg, bool &exc) {
    exc |= fp_is_zero(b.y);
    G1X r;
    r.x = b.x;
    r.y = fp_cond_neg(b.y, neg);
    r.zz = fp_one();
    r.zzz = fp_one();
    return r;
}

// As g1x_madd_acc, but a may be the identity (used where accumulators can
// start empty).
VKZG_DEV G1X g1x_madd_fast(const G1X &a, const G1A &b, bool &exc) {
    if (g1a_is_identity(b)) return a;
    if (fp_is_zero(a.zz)) return g1x_from_affine(b);
    return g1x_madd_acc(a, b, false, exc);
}

// add-2008-s without the identity checks: a and b are not the identity.
// The products are ordered so that every input coordinate dies as early as
// possible (ZZ1 ZZ2 and ZZZ1 ZZZ2 first), which keeps the sum within a
// register budget where two other points are live.
VKZG_DEV G1X g1x_add_core(const G1X &a, const G1X &b, bool &exc) {
    const Fp U1 = fp_mul(a.x, b.zz);
    const Fp P = fp_mul_fold(b.x, a.zz, U1, -1);
    const Fp ZZ12 = fp_mul(a.zz, b.zz);
    const Fp S1 = fp_mul(a.y, b.zzz);
    const Fp R = fp_mul_fold(b.y, a.zzz, S1, -1);
    const Fp ZZZ12 = fp_mul(a.zzz, b.zzz);
    const Fp PP = fp_sqr(P);
    exc |= fp_is_zero(PP);
    return g1x_add_tail(U1, S1, ZZ12, ZZZ12, P, PP, R);
}

// a + b for hot loops (see g1x_madd_acc for the `exc` contract); either may
// be the identity.  Branches rather than selects around the sum, so neither
// input has to stay live to the end.
VKZG_DEV G1X g1x_add_fast(const G1X &a, const G1X &b, bool &exc) {
    G1X r = a;
    if (!fp_is_zero(b.zz)) {
        if (fp_is_zero(a.zz)) r = b;
        else r = g1x_add_core(a, b, exc);
    }
    return r;
}

// add-2008-s: XYZZ + XYZZ
VKZG_DEV_CALL G1X g1x_add(const G1X &a, const G1X &b) {
    if (fp_is_zero(a.zz)) return b;
    if (fp_is_zero(b.zz)) return a;
    const Fp U1 = fp_mul(a.x, b.zz);
    const Fp P = fp_mul_fold(b.x, a.zz, U1, -1);
    const Fp S1 = fp_mul(a.y, b.zzz);
    const Fp R = fp_mul_fold(b.y, a.zzz, S1, -1);
    const Fp PP = fp_sqr(P);
    if (fp_is_zero(PP)) {
        if (fp_is_zero_mod(R)) return g1x_dbl_cold(a);
        return g1x_identity();
    }
    return g1x_add_tail(U1, S1, fp_mul(a.zz, b.zz), fp_mul(a.zzz, b.zzz), P, PP, R);
}

// The four lanes of a quad hold the same point(s) and share one operation:
// its products are split into dependent rounds of at most four, and DPP quad
// broadcasts give every lane each round's products.  The same formulas as
// g1x_dbl (3 rounds instead of 9 products) and g1x_add_fast (4 rounds instead
// of 14).
VKZG_DEV G1X g1x_dbl_quad(const G1X &p, uint32_t q) {
    if (fp_is_zero(p.zz)) return p;  // uniform in the quad
    const bool odd = (q & 1u) != 0;
    const Fp r1 = fp_mul(fp_select(odd, p.x, fp_dbl_raw(p.y)), fp_select(odd, p.x, p.y));
    const Fp V = fp_dbl_raw(fp_quad_bcast<0>(r1));  // 4 Y^2
    const Fp M = fp_triple(fp_quad_bcast<1>(r1));   // 3 X^2
    const Fp r2 = fp_mul(fp_select(q == 2, M, V), fp_select4(q, p.y, p.x, M, p.zz));
    const Fp W = fp_dbl_raw(fp_quad_bcast<0>(r2)), S = fp_quad_bcast<1>(r2);  // 8 Y^3, 4 X Y^2
    G1X r;
    r.x = fp_neg(fp_dbl_sub(S, fp_quad_bcast<2>(r2)));  // M^2 - 2S
    r.zz = fp_quad_bcast<3>(r2);                        // V ZZ
    const Fp r3 = fp_mul(fp_select(q == 0, fp_sub_raw(S, r.x), W), fp_select4(q, M, p.y, p.zzz, p.zzz));
    r.y = fp_sub(fp_quad_bcast<0>(r3), fp_quad_bcast<1>(r3));  // M (S - X3) - W Y
    r.zzz = fp_quad_bcast<2>(r3);                               // W ZZZ
    return r;
}

// Rounds: {U1, U2, S1, S2}, {PP, RR, ZZ1 ZZ2, ZZZ1 ZZZ2}, {PPP, Q, ZZ3, -X3},
// {R (Q - X3), S1 PPP, ZZZ3}.  With PPP + 2Q = (U1 + U2) PP the fourth lane of
// the third round makes -X3 = (U1 + U2) PP - R^2 itself.
VKZG_DEV G1X g1x_add_quad(const G1X &a, const G1X &b, uint32_t q, bool &exc) {
    if (fp_is_zero(a.zz)) return b;  // uniform in the quad
    if (fp_is_zero(b.zz)) return a;
    const Fp r1 = fp_mul(fp_select4(q, a.x, b.x, a.y, b.y), fp_select4(q, b.zz, a.zz, b.zzz, a.zzz));
    const Fp U1 = fp_quad_bcast<0>(r1), U2 = fp_quad_bcast<1>(r1);
    const Fp S1 = fp_quad_bcast<2>(r1), S2 = fp_quad_bcast<3>(r1);
    const Fp P = fp_sub(U2, U1), R = fp_sub(S2, S1);
    const Fp r2 = fp_mul(fp_select4(q, P, R, a.zz, a.zzz), fp_select4(q, P, R, b.zz, b.zzz));
    const Fp PP = fp_quad_bcast<0>(r2), RR = fp_quad_bcast<1>(r2);
    const Fp ZZab = fp_quad_bcast<2>(r2), ZZZab = fp_quad_bcast<3>(r2);
    exc |= fp_is_zero(PP);
    const Fp r3 = fp_mul_fold_v(fp_select4(q, P, U1, ZZab, fp_add_raw(U1, U2)), PP, RR, q == 3 ? -1 : 0);
    const Fp PPP = fp_quad_bcast<0>(r3), Q = fp_quad_bcast<1>(r3), nX = fp_quad_bcast<3>(r3);
    G1X r;
    r.zz = fp_quad_bcast<2>(r3);
    r.x = fp_neg(nX);
    const Fp r4 = fp_mul(fp_select(q == 0, fp_add_raw(Q, nX), PPP), fp_select4(q, R, S1, ZZZab, ZZZab));
    r.y = fp_sub(fp_quad_bcast<0>(r4), fp_quad_bcast<1>(r4));
    r.zzz = fp_quad_bcast<2>(r4);
    return r;
}

// g1x_madd_acc shared by the four lanes of a quad that all hold a, b and
// neg: its products in four dependent rounds -- {P = U2 - X1, R = S2 - Y1,
// U2 + X1}, {P^2, R^2}, {P PP, X1 PP, ZZ1 PP, -X3 = (U2 + X1) PP - R^2},
// {R (Q - X3), Y1 PPP, ZZZ1 PPP} -- instead of ten products in a row.
VKZG_DEV G1X g1x_madd_acc_quad(const G1X &a, const G1A &b, bool neg, uint32_t q, bool &exc) {
    exc |= fp_is_zero(b.y);
    const bool odd = (q & 1u) != 0;
    const Fp by = fp_cond_neg(b.y, neg);
    const Fp r1 = fp_mul_fold_v(fp_select(odd, by, b.x), fp_select(odd, a.zzz, a.zz), fp_select(odd, a.y, a.x),
                              q == 2 ? 1 : -1);
    const Fp P = fp_quad_bcast<0>(r1), R = fp_quad_bcast<1>(r1), V = fp_quad_bcast<2>(r1);
    const Fp r2 = fp_sqr(fp_select(odd, R, P));
    const Fp PP = fp_quad_bcast<0>(r2), RR = fp_quad_bcast<1>(r2);
    exc |= fp_is_zero(PP);
    const Fp r3 = fp_mul_fold_v(fp_select4(q, P, a.x, a.zz, V), PP, RR, q == 3 ? -1 : 0);
    const Fp PPP = fp_quad_bcast<0>(r3), Q = fp_quad_bcast<1>(r3), nX = fp_quad_bcast<3>(r3);
    G1X r;
    r.zz = fp_quad_bcast<2>(r3);
    r.x = fp_neg(nX);
    const Fp r4 = fp_mul(fp_select(q == 0, fp_add_raw(Q, nX), PPP), fp_select4(q, R, a.y, a.zzz, a.zzz));
    r.y = fp_sub(fp_quad_bcast<0>(r4), fp_quad_bcast<1>(r4));  // R (Q - X3) - Y1 PPP
    r.zzz = fp_quad_bcast<2>(r4);
    return r;
}

VKZG_DEV G1X g1x_neg(const G1X &p) {
    G1X r = p;
    r.y = fp_neg(p.y);
    return r;
}

// --------------------------------------------------------------- encoding

// The words of a point that is not the identity: canonical x, y > (p-1)/2.
VKZG_DEV void g1a_compressed_words(uint32_t *w, const FpU &x, bool y_large) {
    uint32_t xw[12];
    fp_to_words(xw, x);
    xw[11] |= y_large ? 0xa0000000u : 0x80000000u;
#pragma unroll
    for (int i = 0; i < 12; i++) w[i] = __builtin_bswap32(xw[11 - i]);
}

// Affine (Montgomery) -> 48-byte ZCash compressed encoding as 12 big-endian
// words: x big-endian, 0x80 compressed flag, 0x20 when y > (p-1)/2, identity
// = 0xc0 followed by zeros (k_compress_proofs.comp:21-46).
VKZG_DEV_CALL void g1a_compress_words(uint32_t *w, const G1A &p) {
    if (g1a_is_identity(p)) {
        w[0] = __builtin_bswap32(0xc0000000u);
#pragma unroll
        for (int i = 1; i < 12; i++) w[i] = 0;
        return;
    }
    g1a_compressed_words(w, fp_to_canonical(p.x), fp_is_lex_largest(fp_to_canonical(p.y)));
}

// 48-byte ZCash compressed encoding (src: its 12 words as stored, 4-byte
// aligned) -> affine.  The identity decodes to (0, 0).  False for a
// malformed encoding: no compression flag, stray bits after the infinity
// flag, x >= p or an x with no point on the curve.  No subgroup check.
VKZG_DEV bool g1a_decompress(G1A &out, const uint32_t *src) {
    uint32_t w[12];
#pragma unroll
    for (int k = 0; k < 12; k++) w[k] = __builtin_bswap32(src[k]);
    const uint32_t b0 = w[0] >> 24;
    bool ok = (b0 & 0x80u) != 0;
    if (b0 & 0x40u) {
        uint32_t rest = w[0] & 0x3fffffffu;
#pragma unroll
        for (int k = 1; k < 12; k++) rest |= w[k];
        out = g1a_identity();
        return ok && rest == 0;
    }
    uint32_t xw[12];
#pragma unroll
    for (int k = 0; k < 12; k++) xw[k] = w[11 - k];
    xw[11] &= 0x1fffffffu;
    const FpU x = fp_from_words(xw);
    if (!fp_limbs_lt_p(x)) ok = false;
    const Fp xm = fp_from_canonical(x);
    const Fp rhs = fp_add(fp_mul(fp_sqr(xm), xm), fp_const(cfp::FOUR_M));
    Fp y = fp_pow_const_window<12>(rhs, cfp::SQRT_EXP);
    if (!fp_eq(fp_sqr(y), rhs)) ok = false;
    const bool want_large = (b0 & 0x20u) != 0;
    if (fp_is_lex_largest(fp_to_canonical(y)) != want_large) y = fp_neg(y);
    out.x = xm;
    out.y = y;
    return ok;
}

}  // namespace vkzg_amd
