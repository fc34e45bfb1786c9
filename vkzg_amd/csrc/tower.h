// Extension-field and G2 arithmetic for the pairing of cell-proof
// verification (the reference has no verifier: include/vkzg.h:14-18; the
// verification equation is the consensus specs' verify_cell_kzg_proof_batch).
//
//   Fp2  = Fp[u]/(u^2 + 1)
//   Fp12 = Fp2[w]/(w^6 - xi), xi = 1 + u; an element is sum_m a_m w^m with
//          a_m in Fp2, held as 12 Fp values, index 2m + e (e = 0: real part).
//   G2 is on the twist E': y^2 = x^3 + 4 xi over Fp2; psi(x, y) =
//   (x w^-2, y w^-3) maps it into E(Fp12).
//
// Fp2 operations run on one lane.  Fp12 products run on a whole workgroup:
// the 144 Fp products a_i * b_j go to 144 lanes at once (one Montgomery
// multiplication of latency instead of 54-144 in sequence), then cross-lane
// exchanges inside each wave (DPP quad broadcasts and an xor tree) combine
// them into the 12 result coefficients.  That keeps the pairing's long
// dependent chain (about 480 Fp12 products) near a millisecond on one CU,
// where a one-lane tower would take over ten.
#pragma once

#include "curve.h"

namespace vkzg_amd {

struct Fp2 {
    Fp c0, c1;
};
struct G2A {
    Fp2 x, y;
};

VKZG_DEV Fp2 fp2_zero() { return {fp_zero(), fp_zero()}; }
VKZG_DEV Fp2 fp2_one() { return {fp_one(), fp_zero()}; }
VKZG_DEV Fp2 fp2_add(const Fp2 &a, const Fp2 &b) { return {fp_add(a.c0, b.c0), fp_add(a.c1, b.c1)}; }
VKZG_DEV Fp2 fp2_sub(const Fp2 &a, const Fp2 &b) { return {fp_sub(a.c0, b.c0), fp_sub(a.c1, b.c1)}; }
VKZG_DEV Fp2 fp2_neg(const Fp2 &a) { return {fp_neg(a.c0), fp_neg(a.c1)}; }
VKZG_DEV Fp2 fp2_reduce(const Fp2 &a) { return {fp_reduce(a.c0), fp_reduce(a.c1)}; }
VKZG_DEV Fp2 fp2_conj(const Fp2 &a) { return {a.c0, fp_neg(a.c1)}; }
VKZG_DEV bool fp2_is_zero(const Fp2 &a) { return fp_is_zero_mod(a.c0) && fp_is_zero_mod(a.c1); }
VKZG_DEV bool fp2_eq(const Fp2 &a, const Fp2 &b) { return fp_eq(a.c0, b.c0) && fp_eq(a.c1, b.c1); }
// Karatsuba: (a0 + a1 u)(b0 + b1 u) = a0 b0 - a1 b1 + ((a0 + a1)(b0 + b1) - a0 b0 - a1 b1) u
VKZG_DEV Fp2 fp2_mul(const Fp2 &a, const Fp2 &b) {
    const Fp t0 = fp_mul(a.c0, b.c0);
    const Fp t1 = fp_mul(a.c1, b.c1);
    const Fp t2 = fp_mul_fold(fp_add_raw(a.c0, a.c1), fp_add(b.c0, b.c1), t0, -1);
    return {fp_sub(t0, t1), fp_sub(t2, t1)};
}
// (a0 + a1 u)^2 = (a0 + a1)(a0 - a1) + 2 a0 a1 u
VKZG_DEV Fp2 fp2_sqr(const Fp2 &a) {
    return {fp_mul(fp_add_raw(a.c0, a.c1), fp_sub(a.c0, a.c1)), fp_mul(fp_dbl_raw(a.c0), a.c1)};
}
VKZG_DEV Fp2 fp2_mul_fp(const Fp2 &a, const Fp &s) { return {fp_mul(a.c0, s), fp_mul(a.c1, s)}; }
// a * xi = (a0 - a1) + (a0 + a1) u
VKZG_DEV Fp2 fp2_mul_xi(const Fp2 &a) { return {fp_sub(a.c0, a.c1), fp_add(a.c0, a.c1)}; }
// 1/a = conj(a) / (a0^2 + a1^2); 0 -> 0
VKZG_DEV Fp2 fp2_inv(const Fp2 &a) {
    const Fp n = fp_add(fp_sqr(a.c0), fp_sqr(a.c1));
    const Fp ni = fp_inv(n);
    return {fp_mul(a.c0, ni), fp_neg(fp_mul(a.c1, ni))};
}
template <int NE>
VKZG_DEV Fp2 fp2_pow_const(const Fp2 &a, const uint32_t (&e)[NE]) {
    Fp2 acc = fp2_one();
#pragma unroll 1
    for (int i = NE - 1; i >= 0; i--) {
        const uint32_t limb = e[i];
#pragma unroll 1
        for (int b = 31; b >= 0; b--) {
            acc = fp2_sqr(acc);
            if ((limb >> b) & 1u) acc = fp2_mul(acc, a);
        }
    }
    return acc;
}

// Square root in Fp2 for p = 3 mod 4 (Adj and Rodriguez-Henriquez, "Square
// root computation over even extension fields", 2014, Algorithm 9):
//   a1 = a^((p-3)/4), alpha = a1^2 a, x0 = a1 a;
//   alpha = -1: x = u x0; otherwise x = (1 + alpha)^((p-1)/2) x0.
// The result is checked by squaring; false when a is not a square.
VKZG_DEV bool fp2_sqrt(Fp2 &out, const Fp2 &a) {
    const Fp2 a1 = fp2_pow_const<12>(a, cfp::P_MINUS_3_DIV_4);
    const Fp2 alpha = fp2_mul(fp2_sqr(a1), a);
    const Fp2 x0 = fp2_mul(a1, a);
    const Fp2 minus_one = {fp_neg(fp_one()), fp_zero()};
    Fp2 x;
    if (fp2_eq(alpha, minus_one)) {
        x = {fp_neg(x0.c1), x0.c0};  // u * x0
    } else {
        const Fp2 b = fp2_pow_const<12>(fp2_add(fp2_one(), alpha), cfp::P_MINUS_1_DIV_2);
        x = fp2_mul(b, x0);
    }
    out = x;
    return fp2_eq(fp2_sqr(x), a);
}

// Sign of the compressed G2 encoding: y is "larger" when y.c1 > (p-1)/2, or
// y.c1 == 0 and y.c0 > (p-1)/2 (the ZCash serialisation of BLS12-381).
VKZG_DEV bool fp2_is_lex_largest(const Fp2 &y) {
    const FpU c1 = fp_to_canonical(y.c1);
    if (!fpu_is_zero(c1)) return fp_is_lex_largest(c1);
    return fp_is_lex_largest(fp_to_canonical(y.c0));
}

// ------------------------------------------------------------ Fp12 in LDS

VKZG_DEV Fp fp_shfl_xor(const Fp &v, int mask) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = __shfl_xor(v.v[i], mask);
    return r;
}

constexpr uint32_t kFp12Threads = 192;  // lanes an Fp12 product uses (blockDim.x >= this)

// dst = a * b for Fp12 values held in LDS (12 Fp each).  Every thread of the
// block calls it (it contains barriers); blockDim.x >= 192.  dst may alias a
// or b.  Lane t works on output power M = t / 32 and on term m1 = (t % 32) / 4
// (terms 6 and 7 of a group are empty): the quad's four lanes multiply
// a_{m1} (times xi when m1 + m2 >= 6: (x + y u) xi = (x - y) + (x + y) u, an
// N2 operand) and b_{m2}, m2 = M - m1 mod 6, component by component, DPP quad
// broadcasts give every lane the four products, lane 0 of the quad forms the
// real and lane 1 the imaginary part of the term, and an xor tree over the
// group's eight quads adds the six terms.  A term's limbs are below 2^30 and
// the sum of two just fits 32 bits, so the tree takes one carry pass after its
// first level and one at its end.  The result is 12 products of magnitude
// c p: operands of up to 9.3p give c <= 2 * 9.3 * 9.3 / 630 + 1/2 < 0.775 and so
// a result below 9.3p again, a valid operand of the next product.
// Operands and result stay in LDS; the partial sums never leave registers.
__device__ __forceinline__ void fp12_mul_lds(Fp *dst, const Fp *a, const Fp *b) {
    const uint32_t t = threadIdx.x;
    const uint32_t M = (t / 32) % 6, m1 = (t % 32) / 4, q = t & 3u;
    const bool term = t < kFp12Threads && m1 < 6;
    const uint32_t m1c = term ? m1 : 0;
    const uint32_t m2 = (M + 6 - m1c) % 6;
    const bool wrap = m1c > M;
    const uint32_t e = q >> 1;
    const Fp x_in = a[2 * m1c + e], x_other = a[2 * m1c + (e ^ 1u)];
    const Fp y_in = b[2 * m2 + (q & 1u)];
    __syncthreads();  // dst may alias a or b
    // wrapped: real part a0 - a1, imaginary part a1 + a0
    const int32_t k = wrap ? (e ? 1 : -1) : 0;
    Fp xs;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) xs.v[i] = x_in.v[i] + k * x_other.v[i];
    const Fp prod = fp_mul(xs, y_in);
    const Fp p00 = fp_quad_bcast<0>(prod), p01 = fp_quad_bcast<1>(prod);
    const Fp p10 = fp_quad_bcast<2>(prod), p11 = fp_quad_bcast<3>(prod);
    Fp v = fp_select(q == 0, fp_sub_raw(p00, p11), fp_add_raw(p01, p10));
    if (!term || q > 1) v = fp_zero();
    v = fp_norm_wide(fp_add_raw(v, fp_shfl_xor(v, 4)));
    v = fp_add_raw(v, fp_shfl_xor(v, 8));
    v = fp_add_raw(v, fp_shfl_xor(v, 16));
    if (t < kFp12Threads && (t % 32) < 2) dst[2 * M + (t % 32)] = fp_norm_wide(v);
    __syncthreads();
}

// The coefficients of an Fp12 product brought below p in magnitude.
__device__ __forceinline__ void fp12_reduce(Fp *a) {
    if (threadIdx.x < 12) a[threadIdx.x] = fp_reduce(a[threadIdx.x]);
    __syncthreads();
}

VKZG_DEV void fp12_set_one(Fp *a, uint32_t t) {
    if (t < 12) a[t] = t == 0 ? fp_one() : fp_zero();
}
// w -> -w: odd powers negated (the p^6-power Frobenius)
VKZG_DEV void fp12_conj_to(Fp *dst, const Fp *a, uint32_t t) {
    if (t < 12) dst[t] = ((t >> 1) & 1u) ? fp_neg(a[t]) : a[t];
}

}  // namespace vkzg_amd
