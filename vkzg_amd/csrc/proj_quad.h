// G1 in homogeneous coordinates on the four lanes of a quad: doubling chains in
// two dependent products per doubling.
//
// A chain of doublings with too few points to fill the chip takes its length
// times the latency of what each doubling waits for.  In Jacobian or XYZZ
// coordinates that is three rounds of products on a quad (g1x_dbl_quad,
// curve.h); the complete formulas for y^2 = x^3 + b in homogeneous coordinates
// (Renes, Costello, Batina, "Complete addition formulas for prime order elliptic
// curves", 2016, algorithms 7 and 9; E(Fp) has odd order, so they hold for every
// point) take two rounds of four:
//   {Y^2, Z^2, 2XY, 2YZ}, {X3, Z3 and the two halves of Y3}.
// They multiply by 3b = 12.  Coordinates on the isomorphic model
//   3 Y^2 Z = 2 X^3 - Z^3,   x = (sigma / nu) X / Z,   y = sigma Y / Z
// with sigma^2 = -12 and nu^3 = 3 sigma / 2 need no such products: with
// T = Y^2, D = Z^2,
//   doubling: X3 = (T + 3D) 2XY, Y3 = (T + 3D)(T - D) - 8DT, Z3 = 8T YZ
//   addition: with t0 = X1X2, t1 = Y1Y2, t2 = Z1Z2, t3 = X1Y2 + X2Y1,
//     t4 = Y1Z2 + Y2Z1, t5 = X1Z2 + X2Z1:
//     X3 = t3 (t1 + t2) + t4 t5, Y3 = (t1 + t2)(t1 - t2) - 2 t0 t5,
//     Z3 = (t1 - t2) t4 + 2 t0 t3.
// The doubling is the same for any scale of X, so a chain that only doubles may
// leave nu out.  The identity is (0 : 1 : 0); X = Y = Z = 0, which is what the
// conversion makes of an XYZZ identity, stays that way under both formulas and
// counts as the identity where only Z is looked at.
//
// Measured, a wave per SIMD: a doubling 3.9 us in three rounds, 2.2 us in two.
#pragma once

#include "curve.h"

namespace vkzg_amd {

// Homogeneous coordinates, the same in every lane of a quad.
struct G1P {
    Fp x, y, z;
};
// A point spread over a quad, as a doubling leaves it: lane 2 holds X, lane 3 Z,
// lanes 0 and 1 two values whose difference is Y.
struct G1PQ {
    Fp r;
};

// The value lane ((CTRL >> 2q) & 3) of the quad holds, in lane q.
template <int CTRL>
VKZG_DEV Fp fp_quad_perm(const Fp &v) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = __builtin_amdgcn_mov_dpp(v.v[i], CTRL, 0xf, 0xf, false);
    return r;
}
constexpr int quad_perm_ctrl(int a, int b, int c, int d) { return a | b << 2 | c << 4 | d << 6; }

// Products (or N values) of every coordinate.
VKZG_DEV G1PQ g1p_spread(const G1P &p, uint32_t q) {
    return G1PQ{fp_select4(q, p.y, fp_zero(), p.x, p.z)};
}
VKZG_DEV Fp g1pq_y(const G1PQ &p) { return fp_sub(fp_quad_bcast<0>(p.r), fp_quad_bcast<1>(p.r)); }
VKZG_DEV G1P g1p_gather(const G1PQ &p) {
    G1P r;
    r.x = fp_quad_bcast<2>(p.r);
    r.y = g1pq_y(p);
    r.z = fp_quad_bcast<3>(p.r);
    return r;
}

VKZG_DEV G1PQ g1pq_dbl(const G1PQ &p, uint32_t q) {
    // {Y Y, Z Z, 2X Y, 2Z Y}
    const Fp y = g1pq_y(p);
    const Fp o = fp_quad_perm<quad_perm_ctrl(3, 3, 2, 3)>(p.r);  // Z, Z, X, Z
    Fp a;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) a.v[i] = (int32_t)((uint32_t)o.v[i] << (q >> 1));
    const Fp r = fp_mul(fp_select(q == 0, y, a), fp_select(q == 1, o, y));
    // (T + 3D) (T - D), 4D 2T, (T + 3D) 2XY, 4T 2YZ: the left factors are
    // u + 3v of products u, v, at most 2^31 - 4 per limb
    const Fp u = fp_quad_perm<quad_perm_ctrl(0, 1, 0, 0)>(r), v = fp_quad_perm<quad_perm_ctrl(1, 1, 1, 0)>(r);
    const Fp w = fp_quad_perm<quad_perm_ctrl(1, 0, 2, 3)>(r);  // D, T
    Fp l, m;
    const int32_t keep = q < 2 ? -1 : 0, flip = q == 0 ? -1 : 0;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) {
        l.v[i] = u.v[i] + 2 * v.v[i] + v.v[i];
        m.v[i] = (q == 1 ? w.v[i] : r.v[i]) + (((w.v[i] ^ flip) - flip) & keep);
    }
    return G1PQ{fp_mul(fp_norm_wide(l), m)};
}

// a + b, complete: three and a half rounds ({t0, t1, t2, t0 + t1 + t3},
// {t4, t5}, and three sums of two products).
VKZG_DEV G1PQ g1p_add_quad(const G1P &a, const G1P &b, uint32_t q) {
    const Fp ra = fp_mul(fp_select4(q, a.x, a.y, a.z, fp_add_raw(a.x, a.y)),
                         fp_select4(q, b.x, b.y, b.z, fp_add(b.x, b.y)));
    const Fp t0 = fp_quad_bcast<0>(ra), t1 = fp_quad_bcast<1>(ra), t2 = fp_quad_bcast<2>(ra);
    const bool odd = (q & 1u) != 0;
    const Fp rb = fp_mul_fold_v(fp_add_raw(fp_select(odd, a.x, a.y), a.z), fp_add(fp_select(odd, b.x, b.y), b.z),
                                fp_add_raw(fp_select(odd, t0, t1), t2), -1);
    const Fp t4 = fp_quad_bcast<0>(rb), t5 = fp_quad_bcast<1>(rb);
    const Fp t3 = fp_norm_wide(fp_sub_raw(fp_quad_bcast<3>(ra), fp_add_raw(t0, t1)));
    const Fp s = fp_add(t1, t2), d = fp_sub(t1, t2), e = fp_dbl(t0);
    // lane 0: d s - e t5 = Y3, lane 2: s t3 + t4 t5 = X3, lane 3: d t4 + e t3 = Z3
    const Fp zero = fp_zero();
    const Fp f0 = fp_select4(q, d, zero, s, d), f1 = fp_select4(q, s, s, t3, t4);
    const Fp g0 = fp_select4(q, fp_neg(e), zero, t4, e), g1 = fp_select(q == 3, t3, t5);
    return G1PQ{fp_mul_sum(f0, f1, g0, g1)};
}

// Conversions.  XYZZ to (X ZZZ : Y ZZ : sigma ZZ ZZZ), two rounds, without nu: for
// chains that only double.
VKZG_DEV G1PQ g1pq_from_xyzz(const G1X &p, uint32_t q) {
    const Fp r = fp_mul(fp_select4(q, p.y, p.zz, p.x, p.zz), fp_select(q == 0, p.zz, p.zzz));
    const Fp z = fp_mul(r, fp_const(cfp::SIGMA_M));
    return G1PQ{fp_select4(q, r, fp_zero(), r, z)};
}
VKZG_DEV G1P g1p_identity() { return G1P{fp_zero(), fp_one(), fp_zero()}; }
// XYZZ by one lane, ready for g1p_add_quad: (nu X ZZZ : Y ZZ : sigma ZZ ZZZ).
VKZG_DEV G1P g1p_from_xyzz_lane(const G1X &p) {
    if (fp_is_zero(p.zz)) return g1p_identity();
    return G1P{fp_mul(fp_mul(p.x, p.zzz), fp_const(cfp::NU_M)), fp_mul(p.y, p.zz),
               fp_mul(fp_mul(p.zz, p.zzz), fp_const(cfp::SIGMA_M))};
}
VKZG_DEV G1PQ g1pq_shfl_xor(const G1PQ &p, int m) {
    G1PQ r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.r.v[i] = __shfl_xor(p.r.v[i], m);
    return r;
}
// An affine point that is not the identity.
VKZG_DEV G1P g1p_from_affine(const G1A &p) {
    return G1P{fp_mul(p.x, fp_const(cfp::NU_M)), p.y, fp_const(cfp::SIGMA_M)};
}

// The check of a point on the curve, by its quad.
//
// P in G1  <=>  phi(P) == [LAMBDA]P with LAMBDA = z^2 - 1, i.e.
// [z^2]P == phi(P) + P.  Sound for every point of E(Fp): phi^2 + phi + 1 = 0,
// so (phi + LAMBDA + 1)(phi - LAMBDA) = -(LAMBDA^2 + LAMBDA + 1) = -r, and
// (phi - LAMBDA)Q = 0 forces [r]Q = 0.  phi(P) + P = -phi^2(P) = (beta^2 x, -y).
// [z^2]P costs two 64-bit chains, whose 126 doublings and 10 additions are the
// time of the check at any batch that leaves SIMDs idle (16,384 points fill
// them): they run on the quad of a point in homogeneous coordinates, 2 rounds of
// products per doubling instead of 9 products in a row on a lane, at 8 products'
// work (proj_quad.h; complete, so points of small order need no case of their
// own).  With 256 to 8,320 points 1.18 -> 0.38 ms.
VKZG_DEV bool g1_in_subgroup(const G1A &p, uint32_t q) {
    if (g1a_is_identity(p)) return true;
    G1P base = g1p_from_affine(p);
    G1PQ a = g1p_spread(base, q);
#pragma unroll 1
    for (int chain = 0; chain < 2; chain++) {
#pragma unroll 1
        for (int i = 62; i >= 0; i--) {
            a = g1pq_dbl(a, q);
            if ((kZAbs >> i) & 1u) a = g1p_add_quad(g1p_gather(a), base, q);
        }
        base = g1p_gather(a);
    }
    // X / Z = nu beta^2 x / sigma, Y / Z = -y / sigma
    const Fp sigma = fp_const(cfp::SIGMA_M);
    const Fp u = fp_mul(p.x, fp_const(cfp::NU_BETA2_M));
    const Fp t = fp_mul(fp_select4(q, base.x, u, base.y, p.y), fp_select((q & 1u) != 0, base.z, sigma));
    return fp_eq(fp_quad_bcast<0>(t), fp_quad_bcast<1>(t)) &&
           fp_is_zero_mod(fp_add_raw(fp_quad_bcast<2>(t), fp_quad_bcast<3>(t)));
}

}  // namespace vkzg_amd
