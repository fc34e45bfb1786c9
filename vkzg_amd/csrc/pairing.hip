// Optimal ate pairing on BLS12-381 for the batch cell-proof check
// e(P1, Q1) e(P2, Q2) == 1 (consensus specs, verify_cell_kzg_proof_batch;
// the reference has no verifier, include/vkzg.h:14-18).
//
// Both G2 points of the check are setup constants, so their Miller-loop lines
// are computed once, in affine coordinates, when the G2 setup is loaded
// (k_g2_lines).  A call then needs only:
//   k_pair_lines  one block per four iterations of the loop: both points' lines
//                 evaluated at P1, P2 and folded into one value;
//   k_pair_final  one block: the Miller accumulation over the 16 groups and the
//                 final exponentiation, with every Fp12 product spread over
//                 144 lanes and every cyclotomic square over 96 (tower.h); the
//                 other blocks are the subgroup checks of the batch's points.
// The chain of Fp12 products is the time of both, ~75 Miller steps, 315
// cyclotomic squares and 40 products: 1141 -> 842 us for k_pair_final, 8 -> 30 us
// for k_pair_lines.
//
// Miller loop over |z| = 0xd201000000010000 from the top bit down: a
// doubling line per bit, an addition line per set bit below the top (63 + 5
// = 68 lines per point).  The line through T with slope lam (slope on the
// twist), evaluated at P = (xP, yP) in E(Fp) and multiplied by w^3:
//   l = (lam xT - yT) - lam xP w^2 + yP w^3.
// The factor w^3 lies in Fp4 and the dropped vertical lines in Fp6; the final
// exponentiation (p^12 - 1)/r kills both.  As in the oracle, the Miller value
// is not inverted for z < 0, which changes no pairing product's equality
// with 1.
//
// Final exponentiation: f^(p^6 - 1) = conj(f) / f, then ^(p^2 + 1) with the
// p^2-Frobenius, then the hard part through
//   3 (p^4 - p^2 + 1)/r = (z - 1)^2 (z + p)(z^2 + p^2 - 1) + 3
// (Hayashida, Hayasaka and Teruya, "Efficient final exponentiation via
// cyclotomic structure for pairings over families of elliptic curves", 2020).
// The result is therefore e(P, Q)^3 in the oracle's convention; a product is
// 1 exactly when its cube is (3 does not divide r).
#include "pairing.h"

#include "proj_quad.h"
#include "proof_common.h"
#include "verify.h"

namespace vkzg_amd {

namespace {

constexpr uint32_t kPairThreads = kFp12Threads;

VKZG_DEV Fp frob2_const(uint32_t m) {
    switch (m) {
        case 0: return fp_const(cfp::FROB2_0);
        case 1: return fp_const(cfp::FROB2_1);
        case 2: return fp_const(cfp::FROB2_2);
        case 3: return fp_const(cfp::FROB2_3);
        case 4: return fp_const(cfp::FROB2_4);
        default: return fp_const(cfp::FROB2_5);
    }
}
VKZG_DEV Fp2 frob1_const(uint32_t m) {
    switch (m) {
        case 0: return {fp_const(cfp::FROB1_0_C0), fp_const(cfp::FROB1_0_C1)};
        case 1: return {fp_const(cfp::FROB1_1_C0), fp_const(cfp::FROB1_1_C1)};
        case 2: return {fp_const(cfp::FROB1_2_C0), fp_const(cfp::FROB1_2_C1)};
        case 3: return {fp_const(cfp::FROB1_3_C0), fp_const(cfp::FROB1_3_C1)};
        case 4: return {fp_const(cfp::FROB1_4_C0), fp_const(cfp::FROB1_4_C1)};
        default: return {fp_const(cfp::FROB1_5_C0), fp_const(cfp::FROB1_5_C1)};
    }
}

// 96-byte compressed G2 (x.c1 then x.c0, big-endian; flags in the top bits
// of the first byte as for G1) -> affine on E'.  inf[i] = 1 for the point at
// infinity; err |= 1 for a malformed encoding or an x with no point.
__global__ void __launch_bounds__(64) k_g2_decompress(G2A *out, uint32_t *inf, const uint8_t *in, uint32_t n, uint32_t *err) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t *src = reinterpret_cast<const uint32_t *>(in + 96ull * i);
    uint32_t w[24];
#pragma unroll
    for (int k = 0; k < 24; k++) w[k] = __builtin_bswap32(src[k]);
    const uint32_t b0 = w[0] >> 24;
    bool bad = (b0 & 0x80u) == 0;
    G2A r;
    r.x = fp2_zero();
    r.y = fp2_zero();
    if (b0 & 0x40u) {
        uint32_t rest = w[0] & 0x3fffffffu;
#pragma unroll
        for (int k = 1; k < 24; k++) rest |= w[k];
        if (rest) bad = true;
        out[i] = r;
        inf[i] = 1;
        if (bad) atomicOr(err, 1u);
        return;
    }
    uint32_t x1w[12], x0w[12];
#pragma unroll
    for (int k = 0; k < 12; k++) {
        x1w[k] = w[11 - k];
        x0w[k] = w[23 - k];
    }
    x1w[11] &= 0x1fffffffu;
    const FpU x1 = fp_from_words(x1w), x0 = fp_from_words(x0w);
    if (!fp_limbs_lt_p(x1) || !fp_limbs_lt_p(x0)) bad = true;
    r.x = {fp_from_canonical(x0), fp_from_canonical(x1)};
    const Fp four = fp_const(cfp::FOUR_M);
    const Fp2 rhs = fp2_add(fp2_mul(fp2_sqr(r.x), r.x), Fp2{four, four});  // x^3 + 4(1 + u)
    Fp2 y;
    if (!fp2_sqrt(y, rhs)) bad = true;
    const bool want_large = (b0 & 0x20u) != 0;
    if (fp2_is_lex_largest(y) != want_large) y = fp2_neg(y);
    r.y = y;
    out[i] = r;
    inf[i] = 0;
    if (bad) atomicOr(err, 1u);
}

// Affine Miller-loop lines of nq points: lines[q][s] = (lam xT - yT, -lam)
// for the 68 steps s in loop order.  One lane per point; err |= 2 on a zero
// denominator (impossible for a point of order r).
__global__ void __launch_bounds__(64) k_g2_lines(Fp2 *lines, const G2A *qs, uint32_t nq, uint32_t *err) {
    const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nq) return;
    const G2A Q = qs[q];
    G2A T = Q;
    Fp2 *out = lines + (size_t)q * 2 * kPairSteps;
    uint32_t s = 0;
    bool bad = false;
#pragma unroll 1
    for (int i = 62; i >= 0; i--) {
        {
            const Fp2 x2 = fp2_sqr(T.x);
            const Fp2 num = fp2_add(fp2_add(x2, x2), x2);
            const Fp2 den = fp2_add(T.y, T.y);
            if (fp2_is_zero(den)) bad = true;
            const Fp2 lam = fp2_mul(num, fp2_inv(den));
            out[2 * s] = fp2_sub(fp2_mul(lam, T.x), T.y);
            out[2 * s + 1] = fp2_neg(lam);
            s++;
            const Fp2 x3 = fp2_sub(fp2_sub(fp2_sqr(lam), T.x), T.x);
            const Fp2 y3 = fp2_sub(fp2_mul(lam, fp2_sub(T.x, x3)), T.y);
            T.x = fp2_reduce(x3);  // x3 and y3 add the last x and y
            T.y = fp2_reduce(y3);
        }
        if ((kZAbs >> i) & 1u) {
            const Fp2 num = fp2_sub(Q.y, T.y);
            const Fp2 den = fp2_sub(Q.x, T.x);
            if (fp2_is_zero(den)) bad = true;
            const Fp2 lam = fp2_mul(num, fp2_inv(den));
            out[2 * s] = fp2_sub(fp2_mul(lam, T.x), T.y);
            out[2 * s + 1] = fp2_neg(lam);
            s++;
            const Fp2 x3 = fp2_sub(fp2_sub(fp2_sqr(lam), T.x), Q.x);
            const Fp2 y3 = fp2_sub(fp2_mul(lam, fp2_sub(T.x, x3)), T.y);
            T.x = fp2_reduce(x3);  // x3 and y3 add the last x and y
            T.y = fp2_reduce(y3);
        }
    }
    if (bad) atomicOr(err, 2u);
}

// Bit i of |z|: an addition line follows the doubling line of iteration i.
VKZG_DEV bool z_bit(int i) { return ((kZAbs >> i) & 1u) != 0; }

// Block g: the Miller accumulation over the kGroupIters iterations of group g
// alone (from the top: iterations 62 - kGroupIters g down), L[g] = prod over them
// of (l1_s(P1) l2_s(P2))^(2^(doublings left in the group)), P2 negated when
// neg2.  A point at infinity contributes the line 1.  The accumulation's 63
// squarings are a chain, its 68 products by lines are not: blocks fold them into
// 16 values side by side (11 to 15 Fp12 products each), which leaves 75 products in
// k_pair_final's chain instead of 131.
__global__ void __launch_bounds__(kPairThreads) k_pair_lines(Fp *L, const Fp2 *lines1, const Fp2 *lines2,
                                                             const G1A *p1, const G1A *p2, uint32_t neg2) {
    __shared__ Fp l[2 * kGroupLines][12], f[12], v[12];
    const uint32_t t = threadIdx.x;
    const int top = 62 - (int)(kGroupIters * blockIdx.x);
    const int low = top >= (int)kGroupIters ? top - (int)kGroupIters + 1 : 0;
    // the group's lines, and those before it
    uint32_t s0 = 0, n = 0;
    for (int i = 62; i >= low; i--) (i > top ? s0 : n) += z_bit(i) ? 2u : 1u;
    if (t < 2 * n) {  // line s0 + t / 2 at P1 (t even) or P2
        const bool second = (t & 1u) != 0;
        const Fp2 *ln = (second ? lines2 : lines1) + 2 * (s0 + t / 2);
        G1A P = second ? *p2 : *p1;
        Fp *d = l[t];
        for (int k = 0; k < 12; k++) d[k] = fp_zero();
        if (g1a_is_identity(P)) {
            d[0] = fp_one();
        } else {
            if (second && neg2) P.y = fp_neg(P.y);
            const Fp2 c0 = ln[0], c2 = ln[1];
            d[0] = c0.c0;
            d[1] = c0.c1;
            d[4] = fp_mul(c2.c0, P.x);
            d[5] = fp_mul(c2.c1, P.x);
            d[6] = P.y;
        }
    }
    __syncthreads();
    uint32_t s = 0;
#pragma unroll 1
    for (int i = top; i >= low; i--) {
        if (s > 0) fp12_mul_lds(f, f, f);
#pragma unroll 1
        for (uint32_t k = z_bit(i) ? 2 : 1; k > 0; k--, s++) {
            fp12_mul_lds(s > 0 ? v : f, l[2 * s], l[2 * s + 1]);
            if (s > 0) fp12_mul_lds(f, f, v);
        }
    }
    if (t < 12) L[(size_t)blockIdx.x * 12 + t] = f[t];
}

// The steps of the final exponentiation on Fp12 values R[0..] in LDS, d = op(a, b).
// A table and a loop over it instead of a call per step: products and powers are
// inlined, and this keeps one copy of each (the kernel is half as long).
enum : uint8_t { kStepMul, kStepPow, kStepConj, kStepFrob1, kStepFrob2 };
enum : uint8_t { rF, rG, rH, rA, rB, rC, rD, kPairRegs };
struct PairStep {
    uint8_t op, d, a, b;
};
static __constant__ PairStep kFinalSteps[] = {
    // easy part: rG = conj(f), rH = 1/(f conj(f)) -> rF = f^((p^6 - 1)(p^2 + 1)), in the cyclotomic subgroup
    {kStepMul, rH, rG, rH},       // 1/f = conj(f) / (f conj(f))
    {kStepMul, rG, rG, rH},       // f^(p^6 - 1)
    {kStepFrob2, rH, rG, 0},
    {kStepMul, rF, rH, rG},
    // hard part: rF^(3 (p^4 - p^2 + 1)/r); conj is the inverse here
    {kStepPow, rA, rF, 0},
    {kStepMul, rA, rA, rF},
    {kStepConj, rA, rA, 0},       // A = F^(z - 1)
    {kStepPow, rB, rA, 0},
    {kStepMul, rB, rB, rA},
    {kStepConj, rB, rB, 0},       // B = A^(z - 1)
    {kStepPow, rC, rB, 0},
    {kStepConj, rC, rC, 0},
    {kStepFrob1, rG, rB, 0},
    {kStepMul, rC, rC, rG},       // C = B^(z + p)
    {kStepPow, rD, rC, 0},
    {kStepPow, rA, rD, 0},        // C^(z^2)
    {kStepFrob2, rG, rC, 0},
    {kStepMul, rA, rA, rG},
    {kStepConj, rG, rC, 0},
    {kStepMul, rA, rA, rG},       // C^(z^2 + p^2 - 1)
    {kStepMul, rG, rF, rF},
    {kStepMul, rG, rG, rF},       // F^3
    {kStepMul, rA, rA, rG},
};

// dst <- conj(src), dst may be src
__device__ __forceinline__ void fp12_conj(Fp *dst, const Fp *src) {
    if (threadIdx.x < 12) fp12_conj_to(dst, src, threadIdx.x);
    __syncthreads();
}
// dst = src^|z| (dst != src) for src in the cyclotomic subgroup; unit: {one, zero} in LDS
__device__ __forceinline__ void fp12_pow_zabs(Fp *dst, const Fp *src, const Fp *unit, const CycTerm &term) {
    if (threadIdx.x < 12) dst[threadIdx.x] = src[threadIdx.x];
    __syncthreads();
#pragma unroll 1
    for (int i = 62; i >= 0; i--) {
        fp12_cyc_sqr_lds(dst, unit, term);
        if (z_bit(i)) fp12_mul_lds(dst, dst, src);
    }
}
__device__ __forceinline__ void fp12_frob1(Fp *dst, const Fp *src) {
    const uint32_t t = threadIdx.x;
    if (t < 6) {
        const Fp2 a = {src[2 * t], src[2 * t + 1]};
        const Fp2 r = fp2_mul(fp2_conj(a), frob1_const(t));
        dst[2 * t] = r.c0;
        dst[2 * t + 1] = r.c1;
    }
    __syncthreads();
}
__device__ __forceinline__ void fp12_frob2(Fp *dst, const Fp *src) {
    const uint32_t t = threadIdx.x;
    if (t < 12) dst[t] = fp_mul(src[t], frob2_const(t >> 1));
    __syncthreads();
}

// Block 0: Miller accumulation over the 16 group products L, final exponentiation,
// status[0] = 1 when the result is 1 (else 0); out12 (may be null) receives
// the result (12 Fp, Montgomery).  Its one chain of products leaves the rest of
// the chip idle, so the other blocks check the membership in G1 of the npts
// points pts (a quad each, 1/3 of the chain's time): err |= kVfyNotInGroup.
__global__ void __launch_bounds__(kPairThreads) k_pair_final(uint32_t *status, Fp *out12, const Fp *L, const G1A *pts,
                                                             uint32_t npts, uint32_t *err) {
    __shared__ Fp R[kPairRegs][12], unit[2];
    __shared__ Fp Ls[kPairGroups * 12];
    __shared__ uint32_t ok;
    const uint32_t t = threadIdx.x;
    if (blockIdx.x > 0) {
        const uint32_t k = (blockIdx.x - 1) * (kPairThreads / 4) + t / 4;
        if (k < npts && !g1_in_subgroup(pts[k], t & 3u)) atomicOr(err, kVfyNotInGroup);
        return;
    }
    for (uint32_t i = t; i < kPairGroups * 12; i += blockDim.x) Ls[i] = L[i];
    if (t < 2) unit[t] = t == 0 ? fp_one() : fp_zero();
    __syncthreads();
    Fp *const f = R[rF], *const g = R[rG], *const h = R[rH], *const A = R[rA];
    if (t < 12) f[t] = Ls[t];
    __syncthreads();
#pragma unroll 1
    for (int i = 62 - (int)kGroupIters; i >= 0; i--) {
        const bool last = i == 0 || (62 - i) % (int)kGroupIters == (int)kGroupIters - 1;  // of its group
#pragma unroll 1
        for (int k = 0; k < (last ? 2 : 1); k++)
            fp12_mul_lds(f, f, k == 0 ? f : Ls + 12 * ((62 - i) / (int)kGroupIters));
    }
    fp12_conj(g, f);
    fp12_mul_lds(h, f, g);  // f conj(f) = n0 + n1 w^2 + n2 w^4 (in Fp6)
    fp12_reduce(h);
    // its inverse in Fp2[v]/(v^3 - xi), v = w^2, a lane per coefficient:
    // c0 = n0^2 - xi n1 n2, c1 = xi n2^2 - n0 n1, c2 = n1^2 - n0 n2, over
    // n0 c0 + xi (n2 c1 + n1 c2)
    if (t < 3) {
        const auto n = [&](uint32_t k) { return Fp2{h[4 * k], h[4 * k + 1]}; };
        const auto xi_if = [](bool c, const Fp2 &v) {
            const Fp2 x = fp2_mul_xi(v);
            return Fp2{fp_select(c, x.c0, v.c0), fp_select(c, x.c1, v.c1)};
        };
        const uint32_t p = (3 - t) % 3;  // n0, n2, n1 beside c0, c1, c2
        const Fp2 sq = xi_if(t == 1, fp2_sqr(n(p)));
        const Fp2 pr = xi_if(t == 0, fp2_mul(n(t == 0 ? 1 : 0), n(t == 1 ? 1 : 2)));
        const Fp2 c = fp2_sub(sq, pr);
        const Fp2 term = xi_if(t > 0, fp2_mul(n(p), c));
        Fp2 den = term;
#pragma unroll
        for (int i = 0; i < kFpLimbs; i++) {  // the three lanes' terms (sums of few, then reduced)
            den.c0.v[i] = __shfl(term.c0.v[i], 0) + __shfl(term.c0.v[i], 1);
            den.c1.v[i] = __shfl(term.c1.v[i], 0) + __shfl(term.c1.v[i], 1);
        }
        den = {fp_norm_wide(den.c0), fp_norm_wide(den.c1)};
#pragma unroll
        for (int i = 0; i < kFpLimbs; i++) {
            den.c0.v[i] += __shfl(term.c0.v[i], 2);
            den.c1.v[i] += __shfl(term.c1.v[i], 2);
        }
        den = {fp_norm_wide(den.c0), fp_norm_wide(den.c1)};
        const Fp2 r = fp2_mul(c, fp2_inv(den));
        h[4 * t] = r.c0;
        h[4 * t + 1] = r.c1;
        h[4 * t + 2] = fp_zero();
        h[4 * t + 3] = fp_zero();
    }
    __syncthreads();
    const CycTerm term = kCycTable.t[t < 96 ? t : 95];
#pragma unroll 1
    for (uint32_t k = 0; k < sizeof(kFinalSteps) / sizeof(PairStep); k++) {
        const PairStep st = kFinalSteps[k];
        Fp *d = R[st.d];
        const Fp *a = R[st.a], *b = R[st.b];
        switch (st.op) {
            case kStepMul: fp12_mul_lds(d, a, b); break;
            case kStepPow: fp12_pow_zabs(d, a, unit, term); break;
            case kStepConj: fp12_conj(d, a); break;
            case kStepFrob1: fp12_frob1(d, a); break;
            default: fp12_frob2(d, a); break;
        }
    }
    if (t == 0) ok = 1;
    __syncthreads();
    if (t < 12) {
        const bool eq = fp_eq(A[t], t == 0 ? fp_one() : fp_zero());
        if (!eq) ok = 0;
        if (out12) out12[t] = A[t];
    }
    __syncthreads();
    if (t == 0) status[0] = ok;
}

__global__ void k_fp_canonical(Fp *a, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = fp_from_digits(fp_to_canonical(a[i]));
}

}  // namespace

hipError_t launch_fp_canonical(Fp *a, uint32_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_fp_canonical, dim3(blocks_for(n, 64)), dim3(64), 0, s, a, n);
    return hipGetLastError();
}

hipError_t launch_g2_decompress(G2A *out, uint32_t *inf, const uint8_t *in, uint32_t n, uint32_t *err,
                                hipStream_t s) {
    hipLaunchKernelGGL(k_g2_decompress, dim3(blocks_for(n, 64)), dim3(64), 0, s, out, inf, in, n, err);
    return hipGetLastError();
}

hipError_t launch_g2_lines(Fp2 *lines, const G2A *qs, uint32_t nq, uint32_t *err, hipStream_t s) {
    hipLaunchKernelGGL(k_g2_lines, dim3(blocks_for(nq, 64)), dim3(64), 0, s, lines, qs, nq, err);
    return hipGetLastError();
}

hipError_t launch_pairing_check(uint32_t *status, Fp *out12, Fp *L, const Fp2 *lines1, const Fp2 *lines2,
                                const G1A *p1, const G1A *p2, bool neg2, const G1A *pts, uint32_t npts,
                                uint32_t *err, hipStream_t s) {
    hipLaunchKernelGGL(k_pair_lines, dim3(kPairGroups), dim3(kPairThreads), 0, s, L, lines1, lines2, p1, p2,
                       neg2 ? 1u : 0u);
    hipLaunchKernelGGL(k_pair_final, dim3(1 + (uint32_t)blocks_for(npts * 4ull, kPairThreads)), dim3(kPairThreads), 0, s,
                       status, out12, L, pts, npts, err);
    return hipGetLastError();
}

}  // namespace vkzg_amd
