// FK20 phase B inputs: doubling ladders of the split-circulant folds of u.
#include <algorithm>

#include "proj_quad.h"
#include "proof_common.h"

namespace vkzg_amd {

namespace {
// g1j_dbl (curve.h) shared by the two lanes of a pair, which both hold p.
// Its products fall into four dependent rounds of at most two -- {X^2, Y^2},
// {W = 2X B, B^2}, {X3 = E^2 - 4W} (computed by both lanes) and
// {E (2W - X3) - 8 B^2, 2Y Z} -- and DPP exchanges hand each round's results
// to both lanes: a doubling waits on two products and two squarings instead
// of four and three.  The sums are folded into the products (field_fp.h), so
// what is left between the rounds is one carry pass each for E = 3 X^2 and
// 2W - X3.
VKZG_DEV G1J g1j_dbl_pair(const G1J &p, uint32_t q) {
    if (fp_is_zero(p.z)) return p;  // uniform in the pair
    const bool odd = q != 0;
    const Fp r1 = fp_sqr(fp_select(odd, p.y, p.x));
    const Fp E = fp_triple(fp_pair_bcast<0>(r1)), B = fp_pair_bcast<1>(r1);
    const Fp r2 = fp_mul(fp_select(odd, B, fp_dbl_raw(p.x)), B);
    const Fp W = fp_pair_bcast<0>(r2);
    G1J r;
    r.x = fp_sqr_fold(E, W, -4);
    // lane 0 multiplies E by 2W - X3 and folds -8 B^2 in, lane 1 2Y by Z
    const Fp r4 = fp_mul_fold_v(fp_select(odd, fp_dbl_raw(p.y), E), fp_select(odd, p.z, fp_dbl_sub(W, r.x)),
                              fp_pair_bcast<1>(r2), odd ? 0 : -8);
    r.y = fp_pair_bcast<0>(r4);
    r.z = fp_pair_bcast<1>(r4);
    return r;
}

// The phase-B points are linear in u, and so are the doublings, so the
// split-circulant folds (k_fold_ladder.comp) are taken before the ladder:
//   F+[i] = u[i] + u[i+64], F-[i] = u[i] - u[i+64] (i < 64),
//   Fc[i] = F+[i] + F+[i+32], Fn[i] = F+[i] - F+[i+32] (i < 32),
// and chain j of a blob doubles f[j] = Fc[j] (j < 32), Fn[j-32] (j < 64),
// F-[j-64] (j >= 64): lad[blob][d][j] = 2^(kDigitBits d) * f[j], d < kLadPos.
// With `splits` = M segments, pair (blob, m, j) starts from the same folds of
// phase A's 2^(kDigitBits start_m) u (u[(blob*M + m)*128 + k], phase A's MSMs with
// their window groups summed), start_m = lad_start(M, m), and writes
// positions [start_m, start_{m+1}).  LANES (2 or 4) lanes share a chain and exit
// together.  While four-lane chains leave SIMDs idle or fill them with one wave
// (ladder_lanes), the chain's length sets the time: quads double in homogeneous
// coordinates (proj_quad.h, without nu) in two rounds of products, and share
// the additions of the folds (flagged ones are redone checked).  Beyond that
// the issue rate does, and pairs double in Jacobian coordinates, whose squares
// make a doubling the cheaper one in instructions (3 squares and 4 products in
// place of 8 products).  Positions hold the chain's own coordinates: (X, Y, Z)
// with x = sigma X / Z, y = sigma Y / Z from quads, Jacobian from pairs.
template <typename Add>
VKZG_DEV G1X ladder_fold(const G1X *u, uint32_t j, Add add) {
    if (j >= 64) return add(u[j - 64], g1x_neg(u[j]));
    const uint32_t i = j & 31u;
    const G1X lo = add(u[i], u[i + 64]);
    const G1X hi = add(u[i + 32], u[i + 96]);
    return add(lo, j < 32 ? hi : g1x_neg(hi));
}

template <int LANES>
__global__ __launch_bounds__(256) void k_ladder(G1J *lad, const G1X *u, uint32_t splits, uint32_t nblobs,
                                                uint32_t force_checked) {
    // A long dependent chain: give these waves issue priority over the
    // throughput kernels of another sub-batch sharing the SIMD.
    __builtin_amdgcn_s_setprio(3);
    const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t g = tid / LANES, q = tid % LANES;
    if (g >= nblobs * 128 * splits) return;
    const uint32_t j = g % 128, m = (g / 128) % splits, blob = g / (128 * splits);
    const G1X *ub = u + (size_t)(blob * splits + m) * 128;
    const uint32_t d0 = lad_start(splits, m), d1 = m + 1 == splits ? kLadPos : lad_start(splits, m + 1);
    G1J *dst = lad + (size_t)blob * kLadPos * 128 + j;
    if constexpr (LANES == 4) {
        bool exc = force_checked != 0;
        G1X f = ladder_fold(ub, j, [&](const G1X &a, const G1X &b) { return g1x_add_quad(a, b, q, exc); });
        // uniform in the quad
        if (exc) f = ladder_fold(ub, j, [](const G1X &a, const G1X &b) { return g1x_add(a, b); });
        G1PQ p = g1pq_from_xyzz(f, q);
#pragma unroll 1
        for (uint32_t d = d0; d < d1; d++) {
            const Fp y = g1pq_y(p);
            if (q == 0) dst[d * 128].y = y;
            else if (q == 2) dst[d * 128].x = p.r;
            else if (q == 3) dst[d * 128].z = p.r;
            if (d + 1 == d1) break;
#pragma unroll 1
            for (uint32_t k = 0; k < kDigitBits; k++) p = g1pq_dbl(p, q);
        }
    } else {
        G1J p = g1j_from_xyzz(ladder_fold(ub, j, [](const G1X &a, const G1X &b) { return g1x_add(a, b); }));
#pragma unroll 1
        for (uint32_t d = d0; d < d1; d++) {
            if (q == 0) {
                dst[d * 128].x = p.x;
                dst[d * 128].z = p.z;
            } else {
                dst[d * 128].y = p.y;
            }
            if (d + 1 == d1) break;
#pragma unroll 1
            for (uint32_t k = 0; k < kDigitBits; k++) p = g1j_dbl_pair(p, q);
        }
    }
}

// The shares of phase A summed per MSM: usum[msm] = sum_k part[msm * shares + k].
// SUMS partial sums per MSM, sum t adding shares t, t + SUMS, ..., then a tree
// of log2(SUMS) levels.  Q = 4 (while SIMDs are idle and this chain of
// additions is the kernel's time): a quad per sum shares each addition
// (g1x_add_quad, four rounds of products instead of fourteen); any flagged
// doubling or cancellation is redone checked by the MSM's first lane.  Q = 1:
// a lane per sum, with the checked additions.  sum_shape picks both.  The
// ladder reads these sums, so its prologue (a dependent chain per group of
// lanes) adds no partials of its own.  An MSM's lanes sit in one wave and leave
// together, so the shuffles only meet lanes that are there.
VKZG_DEV_COLD void sum_groups_checked(G1X *out, const G1X *part, uint32_t groups) {
    G1X acc = g1x_identity();
    for (uint32_t g = 0; g < groups; g++) acc = g1x_add(acc, part[g]);
    *out = acc;
}

template <uint32_t Q, uint32_t SUMS>
__global__ __launch_bounds__(256) void k_sum_groups(G1X *usum, const G1X *part, uint32_t shares, uint32_t nmsm,
                                                    uint32_t force_checked) {
    const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t msm = tid / (SUMS * Q), t = (tid / Q) % SUMS, qd = tid % Q;
    if (msm >= nmsm) return;
    const G1X *p = part + (size_t)msm * shares;
    G1X acc = t < shares ? p[t] : g1x_identity();
    if constexpr (Q == 4) {
        bool exc = force_checked != 0;
#pragma unroll 1
        for (uint32_t k = t + SUMS; k < shares; k += SUMS) acc = g1x_add_quad(acc, p[k], qd, exc);
#pragma unroll 1
        for (uint32_t m = 1; m < SUMS; m <<= 1) acc = g1x_add_quad(acc, g1x_shfl_xor(acc, m * Q), qd, exc);
        // a flag anywhere in the MSM's lanes
        constexpr uint32_t kLanes = SUMS * Q;
        const uint64_t mask = kLanes == 64 ? ~0ull : (1ull << kLanes) - 1;
        if ((__ballot(exc) >> ((threadIdx.x & 63u) / kLanes * kLanes) & mask) != 0) {
            if (t == 0 && qd == 0) sum_groups_checked(&usum[msm], p, shares);
            return;
        }
    } else {
#pragma unroll 1
        for (uint32_t k = t + SUMS; k < shares; k += SUMS) acc = g1x_add(acc, p[k]);
#pragma unroll 1
        for (uint32_t m = 1; m < SUMS; m <<= 1) acc = g1x_add(acc, g1x_shfl_xor(acc, m));
    }
    if (t == 0 && qd == 0) usum[msm] = acc;
}

// phi[k] = (beta x, y) of pts[k]: the endomorphism [lambda], lambda = z^2 - 1
// (the identity (0, 0) maps to itself).
__global__ void k_glv_phi(G1A *phi, const G1A *pts, uint64_t count, uint32_t *queue_b, uint32_t *queue_r) {
    const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0) {  // work counters of phase B and the bucket reduction
        queue_b[0] = 0u;
        queue_r[0] = 0u;
    }
    if (k >= count) return;
    G1A q = pts[k];
    q.x = fp_mul(q.x, fp_const(cfp::BETA_M));
    phi[k] = q;
}

// Small batches: the ladder points (of quads) in XYZZ form for phase B's quad
// additions instead of normalised ones, and their images under the
// endomorphism.  With z = Z / sigma, (X z, Y z^2, z^2, z^3) and (beta X z, ...):
// no inversion, and a quad per point, whose lanes share the seven products in
// three rounds, {z}, {z^2, X z}, {z^3, beta X z, Y z^2}.  Clears the phase-B and
// bucket-reduction work counters, as k_glv_phi does.
__global__ void __launch_bounds__(256) k_ladder_xyzz(G1X *pts, G1X *phi, const G1J *lad, uint64_t count,
                                                     uint32_t *queue_b, uint32_t *queue_r) {
    const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid == 0) {
        queue_b[0] = 0u;
        queue_r[0] = 0u;
    }
    const uint64_t k = tid >> 2;
    const uint32_t q = (uint32_t)tid & 3u;
    if (k >= count) return;
    const G1J p = lad[k];
    const Fp z = fp_mul(p.z, fp_const(cfp::INV_SIGMA_M));
    const Fp r2 = fp_mul(fp_select(q == 1, p.x, z), z);
    const Fp zz = fp_quad_bcast<0>(r2), x = fp_quad_bcast<1>(r2);
    const Fp r3 = fp_mul(fp_select4(q, z, x, p.y, p.y), fp_select(q == 1, fp_const(cfp::BETA_M), zz));
    if (q == 0) {
        pts[k].zz = zz;
        pts[k].zzz = r3;
    } else if (q == 1) {
        pts[k].x = x;
        phi[k].x = r3;
    } else if (q == 2) {
        pts[k].y = r3;
        phi[k].y = r3;
    } else {
        phi[k].zz = zz;
    }
    if (q == 0) phi[k].zzz = r3;
}

}  // namespace

hipError_t launch_ladder_xyzz(G1X *pts, G1X *phi, const G1J *lad, uint64_t count, uint32_t *queue_b,
                              uint32_t *queue_r, hipStream_t s) {
    hipLaunchKernelGGL(k_ladder_xyzz, dim3(blocks_for(count * 4, 256)), dim3(256), 0, s, pts, phi, lad, count,
                       queue_b, queue_r);
    return hipGetLastError();
}

hipError_t launch_ladder(G1J *lad, const G1X *u, uint32_t splits, uint32_t nblobs, uint32_t lanes,
                         uint32_t force_checked, hipStream_t s) {
    // Workgroups of four waves: the dispatcher spreads a workgroup's waves over
    // a CU's four SIMDs, where one-wave workgroups doubled up on some SIMDs
    // while others idled (1.6 ms instead of 0.9 ms for 256 blobs; each wave's
    // chain is issue-bound, so a shared SIMD halves its rate).  Whole groups
    // of LANES lanes fill each 256-thread block.
    const uint64_t threads = nblobs * 128ull * splits * lanes;
    if (lanes == 4)
        hipLaunchKernelGGL(k_ladder<4>, dim3(blocks_for(threads, 256)), dim3(256), 0, s, lad, u, splits, nblobs,
                           force_checked);
    else if (lanes == 2)
        hipLaunchKernelGGL(k_ladder<2>, dim3(blocks_for(threads, 256)), dim3(256), 0, s, lad, u, splits, nblobs,
                           force_checked);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// An addition of the chain takes 7.5 us on a quad and 14 us on a lane with a
// wave per SIMD (measured at 1 to 21 blobs), and in proportion above.  Quads
// do four times the work, so they win while the lanes are few: 16 of them per
// MSM at 1 blob, 8 or 4 at tens of blobs, a lane or two per MSM at 256.
SumShape sum_shape(uint64_t nmsm, uint32_t shares, uint32_t cus) {
    const double simd_lanes = (double)cus * 4 * 64;
    SumShape best{1, 1, 0.0};
    bool have = false;
    for (uint32_t q : {4u, 1u})
        for (uint32_t sums = q == 4 ? 16 : 8; sums >= (q == 4 ? 4u : 1u); sums /= 2) {
            uint32_t adds = (shares + sums - 1) / sums - 1;
            for (uint32_t m = 1; m < sums; m <<= 1) adds++;
            const double us = adds * (q == 4 ? 7.5 : 14.0) * std::max(1.0, nmsm * sums * q / simd_lanes);
            if (!have || us < best.us) best = SumShape{q, sums, us};
            have = true;
        }
    if (shares <= 1) best.us = 0.0;
    return best;
}

hipError_t launch_sum_groups(G1X *usum, const G1X *part, uint32_t shares, uint32_t nmsm, uint32_t cus,
                             uint32_t force_checked, hipStream_t s) {
    auto run = [&](auto kernel, uint32_t lanes) {
        hipLaunchKernelGGL(kernel, dim3(blocks_for((uint64_t)nmsm * lanes, 256)), dim3(256), 0, s, usum, part, shares,
                           nmsm, force_checked);
    };
    const SumShape f = sum_shape(nmsm, shares, cus);
    switch (f.quad * 100 + f.sums) {
        case 416: run(k_sum_groups<4, 16>, 64); break;
        case 408: run(k_sum_groups<4, 8>, 32); break;
        case 404: run(k_sum_groups<4, 4>, 16); break;
        case 108: run(k_sum_groups<1, 8>, 8); break;
        case 104: run(k_sum_groups<1, 4>, 4); break;
        case 102: run(k_sum_groups<1, 2>, 2); break;
        default: run(k_sum_groups<1, 1>, 1); break;
    }
    return hipGetLastError();
}

hipError_t launch_glv_phi(G1A *phi, const G1A *pts, uint64_t count, uint32_t *queue_b, uint32_t *queue_r,
                          hipStream_t s) {
    hipLaunchKernelGGL(k_glv_phi, dim3(blocks_for(count, 256)), dim3(256), 0, s, phi, pts, count, queue_b,
                       queue_r);
    return hipGetLastError();
}

}  // namespace vkzg_amd
