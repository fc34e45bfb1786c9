// BLS12-381 Fp and Fr Montgomery arithmetic for gfx950, held in VGPRs.
//
// Fr: 8 x 32-bit limbs, radix 2^256, canonical results.  Multiplication is
// Montgomery by product scanning (mont_mul below): each 32x32->64 limb
// product is one v_mad_u64_u32 whose carry-out feeds a v_addc_co_u32 into a
// 96-bit column accumulator; r's top limb has a clear top bit, so one
// conditional subtraction finishes.
//
// Fp: 13 signed limbs of 30 bits, radix 2^390 (field_fp.h).
//
// Semantics follow the reference's field library (src/shaders/field.glsl.inc
// :69-297): the same field elements in Montgomery form; byte encodings are
// canonical big-endian.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "constants.h"
#include "field_fp.h"

namespace vkzg_amd {

struct Fr {
    uint32_t v[8];
};

// ------------------------------------------------------------ limb helpers

// r = t - m when t >= m, else t.
template <int N>
VKZG_DEV void reduce_once(uint32_t *r, const uint32_t *t, const uint32_t (&m)[N]) {
    uint32_t d[N];
    uint32_t br = 0;
#pragma unroll
    for (int i = 0; i < N; i++) {
        const uint64_t s = (uint64_t)t[i] - m[i] - br;
        d[i] = (uint32_t)s;
        br = (uint32_t)(s >> 32) & 1u;
    }
#pragma unroll
    for (int i = 0; i < N; i++) r[i] = br ? t[i] : d[i];
}

// acc (64-bit) += x * y and hi += carry-out: v_mad_u64_u32 leaves its carry
// in VCC and v_addc folds it into the third accumulator word, two VALU
// instructions per limb product (the compiler's own lowering of the same
// expression needs five to six).  `y` is an SGPR operand when it is a
// wave-uniform modulus limb.
VKZG_DEV void mac_vv(uint64_t &acc, uint32_t &hi, uint32_t x, uint32_t y) {
    asm("v_mad_u64_u32 %0, vcc, %2, %3, %0\n\tv_addc_co_u32_e32 %1, vcc, 0, %1, vcc"
        : "+v"(acc), "+v"(hi)
        : "v"(x), "v"(y)
        : "vcc");
}
VKZG_DEV void mac_vs(uint64_t &acc, uint32_t &hi, uint32_t x, uint32_t y) {
    asm("v_mad_u64_u32 %0, vcc, %2, %3, %0\n\tv_addc_co_u32_e32 %1, vcc, 0, %1, vcc"
        : "+v"(acc), "+v"(hi)
        : "v"(x), "s"(y)
        : "vcc");
}
// Both products of one FIPS step, a[j] * b[i - j] and m[j] * p[i - j], in one
// block: the compiler separates consecutive asm blocks with an s_nop.
VKZG_DEV void mac_pair(uint64_t &acc, uint32_t &hi, uint32_t x, uint32_t y, uint32_t mx,
                       uint32_t py) {
    asm("v_mad_u64_u32 %0, vcc, %2, %3, %0\n\t"
        "v_addc_co_u32_e32 %1, vcc, 0, %1, vcc\n\t"
        "v_mad_u64_u32 %0, vcc, %4, %5, %0\n\t"
        "v_addc_co_u32_e32 %1, vcc, 0, %1, vcc"
        : "+v"(acc), "+v"(hi)
        : "v"(x), "v"(y), "v"(mx), "s"(py)
        : "vcc");
}

// Fr (mod r) carry chains written out.  The carry of v_add_co/v_addc and the
// borrow of v_sub_co/v_subb pass through VCC, and a VALU carry read of VCC
// needs no wait states; VCC read as a v_cndmask select does, so one s_nop
// (two wait states) sits before the selects.  A VALU instruction reads at
// most one scalar value (VCC, an SGPR or a literal), so r's limbs 2..7 enter
// the borrow chain from VGPRs; limbs 0 and 1 are the inline constants 1 and
// -1.  The compiler's own lowering of the same chains goes through 64-bit
// adds, about twice the instructions.
//
// r = t - r_mod when t >= r_mod, else t (t < 2^256).
VKZG_DEV void fr_reduce_once(uint32_t *r, const uint32_t *t) {
    uint32_t u[8];
    asm("v_subrev_co_u32_e32 %[u0], vcc, 1, %[t0]\n\t"
        "v_subbrev_co_u32_e32 %[u1], vcc, -1, %[t1], vcc\n\t"
        "v_subb_co_u32_e32 %[u2], vcc, %[t2], %[p2], vcc\n\t"
        "v_subb_co_u32_e32 %[u3], vcc, %[t3], %[p3], vcc\n\t"
        "v_subb_co_u32_e32 %[u4], vcc, %[t4], %[p4], vcc\n\t"
        "v_subb_co_u32_e32 %[u5], vcc, %[t5], %[p5], vcc\n\t"
        "v_subb_co_u32_e32 %[u6], vcc, %[t6], %[p6], vcc\n\t"
        "v_subb_co_u32_e32 %[u7], vcc, %[t7], %[p7], vcc\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32_e32 %[r0], %[u0], %[t0], vcc\n\t"
        "v_cndmask_b32_e32 %[r1], %[u1], %[t1], vcc\n\t"
        "v_cndmask_b32_e32 %[r2], %[u2], %[t2], vcc\n\t"
        "v_cndmask_b32_e32 %[r3], %[u3], %[t3], vcc\n\t"
        "v_cndmask_b32_e32 %[r4], %[u4], %[t4], vcc\n\t"
        "v_cndmask_b32_e32 %[r5], %[u5], %[t5], vcc\n\t"
        "v_cndmask_b32_e32 %[r6], %[u6], %[t6], vcc\n\t"
        "v_cndmask_b32_e32 %[r7], %[u7], %[t7], vcc"
        : [r0] "=&v"(r[0]), [r1] "=&v"(r[1]), [r2] "=&v"(r[2]), [r3] "=&v"(r[3]),
          [r4] "=&v"(r[4]), [r5] "=&v"(r[5]), [r6] "=&v"(r[6]), [r7] "=&v"(r[7]),
          [u0] "=&v"(u[0]), [u1] "=&v"(u[1]), [u2] "=&v"(u[2]), [u3] "=&v"(u[3]),
          [u4] "=&v"(u[4]), [u5] "=&v"(u[5]), [u6] "=&v"(u[6]), [u7] "=&v"(u[7])
        : [t0] "v"(t[0]), [t1] "v"(t[1]), [t2] "v"(t[2]), [t3] "v"(t[3]), [t4] "v"(t[4]),
          [t5] "v"(t[5]), [t6] "v"(t[6]), [t7] "v"(t[7]), [p2] "v"(cfr::P[2]),
          [p3] "v"(cfr::P[3]), [p4] "v"(cfr::P[4]), [p5] "v"(cfr::P[5]), [p6] "v"(cfr::P[6]),
          [p7] "v"(cfr::P[7])
        : "vcc");
}

// r = a + b mod r_mod for a, b < r_mod (a + b < 2^256: no carry out).
VKZG_DEV void fr_add_limbs(uint32_t *r, const uint32_t *a, const uint32_t *b) {
    uint32_t t[8];
    asm("v_add_co_u32_e32 %[t0], vcc, %[a0], %[b0]\n\t"
        "v_addc_co_u32_e32 %[t1], vcc, %[a1], %[b1], vcc\n\t"
        "v_addc_co_u32_e32 %[t2], vcc, %[a2], %[b2], vcc\n\t"
        "v_addc_co_u32_e32 %[t3], vcc, %[a3], %[b3], vcc\n\t"
        "v_addc_co_u32_e32 %[t4], vcc, %[a4], %[b4], vcc\n\t"
        "v_addc_co_u32_e32 %[t5], vcc, %[a5], %[b5], vcc\n\t"
        "v_addc_co_u32_e32 %[t6], vcc, %[a6], %[b6], vcc\n\t"
        "v_addc_co_u32_e32 %[t7], vcc, %[a7], %[b7], vcc"
        : [t0] "=&v"(t[0]), [t1] "=&v"(t[1]), [t2] "=&v"(t[2]), [t3] "=&v"(t[3]),
          [t4] "=&v"(t[4]), [t5] "=&v"(t[5]), [t6] "=&v"(t[6]), [t7] "=&v"(t[7])
        : [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2]), [a3] "v"(a[3]), [a4] "v"(a[4]),
          [a5] "v"(a[5]), [a6] "v"(a[6]), [a7] "v"(a[7]), [b0] "v"(b[0]), [b1] "v"(b[1]),
          [b2] "v"(b[2]), [b3] "v"(b[3]), [b4] "v"(b[4]), [b5] "v"(b[5]), [b6] "v"(b[6]),
          [b7] "v"(b[7])
        : "vcc");
    fr_reduce_once(r, t);
}

// r = a - b mod r_mod for a, b < r_mod: the difference, plus r_mod masked by
// the final borrow.
VKZG_DEV void fr_sub_limbs(uint32_t *r, const uint32_t *a, const uint32_t *b) {
    uint32_t t[8], mask, c;
    asm("v_sub_co_u32_e32 %[t0], vcc, %[a0], %[b0]\n\t"
        "v_subb_co_u32_e32 %[t1], vcc, %[a1], %[b1], vcc\n\t"
        "v_subb_co_u32_e32 %[t2], vcc, %[a2], %[b2], vcc\n\t"
        "v_subb_co_u32_e32 %[t3], vcc, %[a3], %[b3], vcc\n\t"
        "v_subb_co_u32_e32 %[t4], vcc, %[a4], %[b4], vcc\n\t"
        "v_subb_co_u32_e32 %[t5], vcc, %[a5], %[b5], vcc\n\t"
        "v_subb_co_u32_e32 %[t6], vcc, %[a6], %[b6], vcc\n\t"
        "v_subb_co_u32_e32 %[t7], vcc, %[a7], %[b7], vcc\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32_e64 %[m], 0, -1, vcc"
        : [t0] "=&v"(t[0]), [t1] "=&v"(t[1]), [t2] "=&v"(t[2]), [t3] "=&v"(t[3]),
          [t4] "=&v"(t[4]), [t5] "=&v"(t[5]), [t6] "=&v"(t[6]), [t7] "=&v"(t[7]), [m] "=&v"(mask)
        : [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2]), [a3] "v"(a[3]), [a4] "v"(a[4]),
          [a5] "v"(a[5]), [a6] "v"(a[6]), [a7] "v"(a[7]), [b0] "v"(b[0]), [b1] "v"(b[1]),
          [b2] "v"(b[2]), [b3] "v"(b[3]), [b4] "v"(b[4]), [b5] "v"(b[5]), [b6] "v"(b[6]),
          [b7] "v"(b[7])
        : "vcc");
    asm("v_and_b32_e32 %[c], 1, %[m]\n\t"
        "v_add_co_u32_e32 %[r0], vcc, %[c], %[t0]\n\t"
        "v_addc_co_u32_e32 %[r1], vcc, %[m], %[t1], vcc\n\t"
        "v_and_b32_e32 %[c], 0xfffe5bfe, %[m]\n\t"
        "v_addc_co_u32_e32 %[r2], vcc, %[c], %[t2], vcc\n\t"
        "v_and_b32_e32 %[c], 0x53bda402, %[m]\n\t"
        "v_addc_co_u32_e32 %[r3], vcc, %[c], %[t3], vcc\n\t"
        "v_and_b32_e32 %[c], 0x09a1d805, %[m]\n\t"
        "v_addc_co_u32_e32 %[r4], vcc, %[c], %[t4], vcc\n\t"
        "v_and_b32_e32 %[c], 0x3339d808, %[m]\n\t"
        "v_addc_co_u32_e32 %[r5], vcc, %[c], %[t5], vcc\n\t"
        "v_and_b32_e32 %[c], 0x299d7d48, %[m]\n\t"
        "v_addc_co_u32_e32 %[r6], vcc, %[c], %[t6], vcc\n\t"
        "v_and_b32_e32 %[c], 0x73eda753, %[m]\n\t"
        "v_addc_co_u32_e32 %[r7], vcc, %[c], %[t7], vcc"
        : [r0] "=&v"(r[0]), [r1] "=&v"(r[1]), [r2] "=&v"(r[2]), [r3] "=&v"(r[3]),
          [r4] "=&v"(r[4]), [r5] "=&v"(r[5]), [r6] "=&v"(r[6]), [r7] "=&v"(r[7]), [c] "=&v"(c)
        : [t0] "v"(t[0]), [t1] "v"(t[1]), [t2] "v"(t[2]), [t3] "v"(t[3]), [t4] "v"(t[4]),
          [t5] "v"(t[5]), [t6] "v"(t[6]), [t7] "v"(t[7]), [m] "v"(mask)
        : "vcc");
}

// Montgomery multiplication by finely integrated product scanning (FIPS):
// column k of a*b and of m*p are summed together in a 96-bit accumulator,
// m_k = low word * n0 makes the low word vanish, and the accumulator shifts
// down one word per column.  Inputs below the modulus give a result below
// twice the modulus (the modulus' top bit is clear), reduced once.
template <int N>
VKZG_DEV void mont_mul(uint32_t *r, const uint32_t *a, const uint32_t *b, const uint32_t (&p)[N],
                       uint32_t n0) {
    uint32_t m[N];
    uint64_t acc = 0;
    uint32_t hi = 0;
#pragma unroll
    for (int i = 0; i < N; i++) {
#pragma unroll
        for (int j = 0; j < i; j++) mac_pair(acc, hi, a[j], b[i - j], m[j], p[i - j]);
        mac_vv(acc, hi, a[i], b[0]);
        m[i] = (uint32_t)acc * n0;
        mac_vs(acc, hi, m[i], p[0]);
        acc = (acc >> 32) | ((uint64_t)hi << 32);
        hi = 0;
    }
    uint32_t t[N];
#pragma unroll
    for (int i = N; i < 2 * N; i++) {
#pragma unroll
        for (int j = i - N + 1; j < N; j++) mac_pair(acc, hi, a[j], b[i - j], m[j], p[i - j]);
        t[i - N] = (uint32_t)acc;
        acc = (acc >> 32) | ((uint64_t)hi << 32);
        hi = 0;
    }
    if constexpr (N == 8) {
        fr_reduce_once(r, t);
    } else {
        reduce_once<N>(r, t, p);
    }
}

// The same product by operand scanning (CIOS) in plain C++; the test hooks
// compute both forms and flag any disagreement.
template <int N>
VKZG_DEV void mont_mul_cios(uint32_t *r, const uint32_t *a, const uint32_t *b,
                            const uint32_t (&m)[N], uint32_t n0) {
    uint32_t t[N];
#pragma unroll
    for (int j = 0; j < N; j++) t[j] = 0;
#pragma unroll
    for (int i = 0; i < N; i++) {
        const uint32_t bi = b[i];
        uint64_t s = (uint64_t)a[0] * bi + t[0];
        t[0] = (uint32_t)s;
        uint32_t A = (uint32_t)(s >> 32);
        const uint32_t mm = t[0] * n0;
        uint64_t q = (uint64_t)mm * m[0] + t[0];
        uint32_t C = (uint32_t)(q >> 32);
#pragma unroll
        for (int j = 1; j < N; j++) {
            s = (uint64_t)a[j] * bi + t[j] + A;
            t[j] = (uint32_t)s;
            A = (uint32_t)(s >> 32);
            q = (uint64_t)mm * m[j] + t[j] + C;
            t[j - 1] = (uint32_t)q;
            C = (uint32_t)(q >> 32);
        }
        t[N - 1] = C + A;
    }
    reduce_once<N>(r, t, m);
}

template <int N>
VKZG_DEV bool limbs_eq(const uint32_t *a, const uint32_t *b) {
    uint32_t acc = 0;
#pragma unroll
    for (int i = 0; i < N; i++) acc |= a[i] ^ b[i];
    return acc == 0;
}

// a < m as plain integers
template <int N>
VKZG_DEV bool limbs_lt(const uint32_t *a, const uint32_t (&m)[N]) {
    uint32_t br = 0;
#pragma unroll
    for (int i = 0; i < N; i++) {
        const uint64_t s = (uint64_t)a[i] - m[i] - br;
        br = (uint32_t)(s >> 32) & 1u;
    }
    return br != 0;
}

// ------------------------------------------------------------------ Fr

VKZG_DEV Fr fr_zero() {
    Fr r;
#pragma unroll
    for (int i = 0; i < 8; i++) r.v[i] = 0;
    return r;
}
VKZG_DEV Fr fr_one() {
    Fr r;
#pragma unroll
    for (int i = 0; i < 8; i++) r.v[i] = cfr::ONE[i];
    return r;
}
VKZG_DEV Fr fr_const(const uint32_t (&c)[8]) {
    Fr r;
#pragma unroll
    for (int i = 0; i < 8; i++) r.v[i] = c[i];
    return r;
}
VKZG_DEV Fr fr_mul(const Fr &a, const Fr &b) {
    Fr r;
    mont_mul<8>(r.v, a.v, b.v, cfr::P, cfr::N0);
    return r;
}
VKZG_DEV Fr fr_sqr(const Fr &a) { return fr_mul(a, a); }
VKZG_DEV Fr fr_add(const Fr &a, const Fr &b) {
    Fr r;
    fr_add_limbs(r.v, a.v, b.v);
    return r;
}
VKZG_DEV Fr fr_sub(const Fr &a, const Fr &b) {
    Fr r;
    fr_sub_limbs(r.v, a.v, b.v);
    return r;
}
VKZG_DEV Fr fr_neg(const Fr &a) { return fr_sub(fr_zero(), a); }

// Montgomery -> canonical (multiply by plain 1).
VKZG_DEV Fr fr_to_canonical(const Fr &a) {
    Fr one = fr_zero();
    one.v[0] = 1;
    return fr_mul(a, one);
}
// canonical (< r) -> Montgomery.
VKZG_DEV Fr fr_from_canonical(const Fr &a) { return fr_mul(a, fr_const(cfr::R2)); }
// Any 256-bit value -> Montgomery form of (value mod r).  2^256 < 3r, so at
// most two subtractions bring it below r first (k_cells_to_fr.comp:5-6 reduces
// non-canonical cell bytes mod r).
VKZG_DEV Fr fr_from_any(const Fr &a) {
    Fr t;
    fr_reduce_once(t.v, a.v);
    fr_reduce_once(t.v, t.v);
    return fr_from_canonical(t);
}

template <int NE>
VKZG_DEV Fr fr_pow_const(const Fr &a, const uint32_t (&e)[NE]) {
    Fr acc = fr_one();
#pragma unroll 1
    for (int i = NE - 1; i >= 0; i--) {
        const uint32_t limb = e[i];
#pragma unroll 1
        for (int b = 31; b >= 0; b--) {
            acc = fr_sqr(acc);
            if ((limb >> b) & 1u) acc = fr_mul(acc, a);
        }
    }
    return acc;
}
VKZG_DEV Fr fr_inv(const Fr &a) { return fr_pow_const<8>(a, cfr::P_MINUS_2); }

// 32 big-endian bytes (as 8 big-endian words) -> little-endian limbs
// A canonical a < r as sign and magnitude: r - a with bit 255 set when
// r - a < a, else a.  The magnitude is at most (r - 1) / 2 < 2^254; bit 255 is
// free since r < 2^255.
VKZG_DEV Fr fr_signed_magnitude(const Fr &a) {
    Fr n;
    uint32_t br = 0, lt = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint64_t d = (uint64_t)cfr::P[i] - a.v[i] - br;
        n.v[i] = (uint32_t)d;
        br = (uint32_t)(d >> 32) & 1u;
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint64_t d = (uint64_t)n.v[i] - a.v[i] - lt;
        lt = (uint32_t)(d >> 32) & 1u;
    }
    if (!lt) return a;
    n.v[7] |= 0x80000000u;
    return n;
}
VKZG_DEV Fr fr_from_be_words(const uint32_t *w) {
    Fr r;
#pragma unroll
    for (int i = 0; i < 8; i++) r.v[i] = __builtin_bswap32(w[7 - i]);
    return r;
}
VKZG_DEV void fr_to_be_words(uint32_t *w, const Fr &a) {
#pragma unroll
    for (int i = 0; i < 8; i++) w[7 - i] = __builtin_bswap32(a.v[i]);
}

// ------------------------------------------------------ Fp across lanes

// The value lane k of this lane's quad holds (DPP quad_perm [k,k,k,k]), word
// by word; the quad's four lanes must all be active.
template <int K>
VKZG_DEV Fp fp_quad_bcast(const Fp &v) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++)
        r.v[i] = __builtin_amdgcn_mov_dpp(v.v[i], K * 0x55, 0xf, 0xf, false);
    return r;
}

// The value lane k of this lane's pair (lanes 2i, 2i+1) holds (DPP quad_perm
// [0,0,2,2] or [1,1,3,3]); both lanes of the pair must be active.
template <int K>
VKZG_DEV Fp fp_pair_bcast(const Fp &v) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++)
        r.v[i] = __builtin_amdgcn_mov_dpp(v.v[i], K ? 0xF5 : 0xA0, 0xf, 0xf, false);
    return r;
}

}  // namespace vkzg_amd
