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
// exchanges inside each wave (DPP quad broadcasts and a tree) combine them into
// the 12 result coefficients.  That keeps the pairing's long dependent chain
// (about 115 Fp12 products and 315 cyclotomic squares) below a millisecond on
// one CU, where a one-lane tower would take over ten.
#pragma once

#include "curve.h"
#include "fp12_tree.h"

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

constexpr uint32_t kFp12Threads = 192;  // lanes an Fp12 product uses (blockDim.x >= this)

// dst = a * b for Fp12 values held in LDS (12 Fp each).  Every thread of the
// block calls it (it contains barriers); blockDim.x >= 192.  dst may alias a
// or b.  Lane t works on output power M = t / 32 and on term m1 of it, four lanes
// to a term (fp12_term): the quad's lanes multiply
// a_{m1} (times xi when m1 + m2 >= 6: (x + y u) xi = (x - y) + (x + y) u, an
// N2 operand) and b_{m2}, m2 = M - m1 mod 6, component by component, DPP quad
// broadcasts give every lane the four products, lane 0 of the quad forms the
// real and lane 1 the imaginary part of the term, and a tree over the group's
// quads (fp12_tree) adds the six terms.  The result is 12 products of magnitude
// c p: operands of up to 12.3p give c <= 2 * 12.3 * 12.3 / 630 + 1/2 < 0.981 and
// so a result below 11.8p, a valid operand of the next product or square.
// Operands and result stay in LDS; the partial sums never leave registers.
__device__ __forceinline__ void fp12_mul_lds(Fp *dst, const Fp *a, const Fp *b) {
    const uint32_t t = threadIdx.x;
    const uint32_t M = (t / 32) % 6, q = t & 3u;
    const bool term = t < kFp12Threads && fp12_has_term(t);
    const uint32_t m1 = term ? fp12_term(t) : 0;
    const uint32_t m2 = (M + 6 - m1) % 6;
    const bool wrap = m1 > M;
    const uint32_t e = q >> 1;
    const Fp x_in = a[2 * m1 + e], x_other = a[2 * m1 + (e ^ 1u)];
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
    v = fp12_tree(v);
    if (t < kFp12Threads && (t % 32) < 2) dst[2 * M + (t % 32)] = v;
    __syncthreads();
}

// Squares in the cyclotomic subgroup (Granger and Scott, "Faster squaring in the
// cyclotomic subgroup of sixth degree extensions", 2010): with a = A + B w + C w^2
// over Fp4 = Fp2[s]/(s^2 - xi), s = w^3, and bar: s -> -s,
//   a^2 = (3 A^2 - 2 bar A) + (3 s C^2 + 2 bar B) w + (3 B^2 - 2 bar C) w^2.
// Each of the 12 coefficients is then 3 times a sum of at most five products of
// two coefficients of a (one of them doubled in some), plus or minus 2 z for one
// coefficient z: eight lanes per coefficient, the sum of lanes 0 to 2 and 4 to 6
// and, on lane 7, z times 1, which keeps z from growing -- 96 lanes, plain products
// of values in LDS, and DPP within a row where the general product has 144 lanes,
// operands to prepare and a tree over 32 lanes.  A square takes 1.6 us
// where the general product takes 2.2.
struct CycTerm {
    uint8_t a, b;      // operands: 0..11 a coefficient, 12 one, 13 zero
    uint8_t dbl, neg;  // +-(2a or a) b
};
struct CycTable {
    CycTerm t[96];
};
constexpr CycTable cyc_table() {
    CycTable r{};
    for (int o = 0; o < 12; o++) {
        const int m = o / 2, e = o % 2;
        // x, y: the two coefficients squared or multiplied
        const int x0 = 2 * (m == 0 || m == 3 ? 0 : (m == 1 || m == 4 ? 2 : 1)), x1 = x0 + 1;
        const int y0 = x0 + 6, y1 = y0 + 1;
        CycTerm *t = r.t + 8 * o;
        for (int k = 0; k < 8; k++) t[k] = {13, 13, 0, 0};
        t[7] = {(uint8_t)o, 12, 0, 0};
        auto set = [&](int k, int a, int b, int dbl, int neg) {
            t[k] = {(uint8_t)a, (uint8_t)b, (uint8_t)dbl, (uint8_t)neg};
        };
        if (m % 2 == 0) {  // x^2 + xi y^2 (xi y^2: (Re - Im, Re + Im) of y^2)
            if (e == 0) set(0, x0, x0, 0, 0), set(1, x1, x1, 0, 1), set(5, y0, y1, 1, 1);
            else set(0, x0, x1, 1, 0), set(5, y0, y1, 1, 0);
            set(2, y0, y0, 0, 0), set(4, y1, y1, 0, 1);
        } else if (m != 1) {  // 2 x y
            if (e == 0) set(0, x0, y0, 1, 0), set(1, x1, y1, 1, 1);
            else set(0, x0, y1, 1, 0), set(1, x1, y0, 1, 0);
        } else {  // 2 xi x y
            set(0, x0, y0, 1, 0), set(1, x1, y1, 1, 1);
            set(4, x0, y1, 1, e ? 0 : 1), set(5, x1, y0, 1, e ? 0 : 1);
        }
    }
    return r;
}
static __constant__ CycTable kCycTable = cyc_table();

// a <- a^2 for a in the cyclotomic subgroup, in LDS; unit: {one, zero} there.
// Every thread of the block calls it; t: this thread's term (unused from 96 up).
// With coefficients of up to 12.3p a result is below 10.8p: at most 3 (3 or 4
// times 12.3^2 / 630) for the exact values of the sums (|x0^2 - x1^2| <= z^2,
// |y0^2 - y1^2 -+ 2 y0 y1| <= 2 z^2, twice |x y xi| <= 4 z^2), 3 (5/2 or 4/2) for the
// products' roundings and 2 (12.3 / 630 + 1/2) for z.
__device__ __forceinline__ void fp12_cyc_sqr_lds(Fp *a, const Fp *unit, const CycTerm &term) {
    const uint32_t t = threadIdx.x, o = (t / 8) % 12, m = o / 2;
    Fp x = *(term.a < 12 ? a + term.a : unit + (term.a - 12));
    const Fp y = *(term.b < 12 ? a + term.b : unit + (term.b - 12));
    __syncthreads();
    if (t < 96) {
#pragma unroll
        for (int i = 0; i < kFpLimbs; i++) x.v[i] = (int32_t)((uint32_t)x.v[i] << term.dbl);
        const Fp p = fp_mul(x, y);
        const Fp s = fp_cond_neg(p, term.neg != 0);
        // lanes 0 and 4: the sums of three; lane 0 then takes lane 4's and lane 7's product
        const Fp s3 = fp_add_raw(fp_add_raw(s, fp_row_dpp<kRowShl + 1>(s)), fp_row_dpp<kRowShl + 2>(s));
        const Fp s6 = fp_row_dpp<kRowShl + 4>(s3), z = fp_row_dpp<kRowShl + 7>(p);
        const int32_t G = m % 2 ? 2 : -2;
        if ((t & 7u) == 0) {
            const int32_t three = fp_hidden(3);
            int64_t acc = 0;
            Fp r;
#pragma unroll
            for (int i = 0; i < kFpLimbs; i++) {
                fp_mac(acc, s3.v[i], three);
                fp_mac(acc, s6.v[i], three);
                fp_mac(acc, z.v[i], G);
                if (i + 1 < kFpLimbs) {
                    r.v[i] = fp_digit((uint32_t)acc);
                    acc = (acc + (1 << (kFpBits - 1))) >> kFpBits;
                    fp_hide(acc);
                } else {
                    r.v[i] = (int32_t)acc;
                }
            }
            a[o] = r;
        }
    }
    __syncthreads();
}

// The coefficients of an Fp12 product brought below p in magnitude.
__device__ __forceinline__ void fp12_reduce(Fp *a) {
    if (threadIdx.x < 12) a[threadIdx.x] = fp_reduce(a[threadIdx.x]);
    __syncthreads();
}

// w -> -w: odd powers negated (the p^6-power Frobenius)
VKZG_DEV void fp12_conj_to(Fp *dst, const Fp *a, uint32_t t) {
    if (t < 12) dst[t] = ((t >> 1) & 1u) ? fp_neg(a[t]) : a[t];
}

}  // namespace vkzg_amd
