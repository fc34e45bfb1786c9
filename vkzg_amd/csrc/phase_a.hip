// FK20 phase A: 128 fixed-base MSMs of length 64 per blob (see kernels.h).
#include "proof_common.h"

namespace vkzg_amd {

namespace {
// Phase-A scalars come as sign (bit 255) and magnitude plus scalar_bias
// (k_fk20_scalars): with the bias of (half - 1) 2^bit(w) in every window below
// the top one, the window's bits are its signed digit plus half - 1, so no
// carry comes up from the windows below.  The digit of window w from the
// window's bits: its magnitude, and in neg its sign times the scalar's.
VKZG_DEV uint32_t window_digit(uint32_t raw, const WindowPlan &plan, uint32_t w, bool sneg, bool &neg) {
    const int32_t d = (int32_t)raw - (w + 1 < plan.W ? (int32_t)((plan.H() << plan.wide(w)) - 1u) : 0);
    neg = (d < 0) != sneg;
    return (uint32_t)(d < 0 ? -d : d);
}

// A scalar whose low bits are the bits of the window at hand.  Windows are
// uniform in a wave, so stepping to the next one is eight funnel shifts.
struct ScalarBits {
    Fr v;
    bool neg;
    VKZG_DEV void load(const Fr &s) {
        v = s;
        neg = (s.v[7] >> 31) != 0;
        v.v[7] &= 0x7fffffffu;
    }
    VKZG_DEV void skip(uint32_t bits) {
#pragma unroll 1
        for (; bits >= 32; bits -= 32) {
#pragma unroll
            for (int i = 0; i < 7; i++) v.v[i] = v.v[i + 1];
            v.v[7] = 0;
        }
#pragma unroll
        for (int i = 0; i < 7; i++) v.v[i] = __builtin_amdgcn_alignbit(v.v[i + 1], v.v[i], bits);
        v.v[7] >>= bits;
    }
    VKZG_DEV uint32_t low(uint32_t width) const { return v.v[0] & ((1u << width) - 1u); }
};

// Windows [w0, w1) of `terms` terms of one MSM, recomputed with the checked
// point operations: reached only when the fast path flagged a doubling or
// cancellation case in this lane's share.
__device__ __attribute__((noinline)) void phase_a_slow(G1X *out, const Fr *scal, const G1AT *tab, WindowPlan plan,
                                                       uint32_t terms, uint32_t w0, uint32_t w1) {
    G1X acc = g1x_identity();
#pragma unroll 1
    for (uint32_t i = 0; i < terms; i++) {
        ScalarBits s;
        s.load(scal[i]);
        s.skip(plan.bit(w0));
        const G1AT *row = tab + (size_t)i * plan.entries();
#pragma unroll 1
        for (uint32_t w = w0; w < w1; w++) {
            const uint32_t width = plan.c + plan.wide(w);
            bool neg;
            const uint32_t mag = window_digit(s.low(width), plan, w, s.neg, neg);
            s.skip(width);
            if (mag) acc = g1x_madd(acc, g1a_neg_if(row[plan.entry(w) + (mag - 1)].p, neg));
        }
    }
    *out = acc;
}

// Persistent phase A.  MSM m = (blob * splits + seg) * nj + j, j < nj, is
//   u[m] = sum_{i<64} scal[m][i] * base[j][i]
// (nj = 128 and the bases x_ext_fft for the proofs; nj = 64 and the setup's
// 4096 points for commitments)
// with the scalar in signed digits v in [-(2^(b-1)-1), 2^(b-1)] of each window's
// width b (the recoding of k_phase_a_sort.comp:31-40 with the plan's windows),
// each digit's sign flipped for a negative scalar, and
// table[j][i][entry(w) + |v| - 1] = |v| * 2^bit(w) * base[j][i].  Its terms are
// cut into `parts` runs of 64 / parts and its windows into `groups` groups, and
// one lane adds up one (run, group) share: part[m * parts * groups + share].
// k_sum_groups adds an MSM's shares.
//
// A wave's 64 lanes are 64 MSMs of one share, in the order (j, seg, blob) with
// the blob fastest: they run the same windows of the same terms, and from 64
// blobs on also against the same base, so that their random 128-byte lines
// lie in one megabyte of the table.  A wave over 8 bases and 8 runs of terms,
// with a lane tree over the runs, gathered from 64 such places at once and
// spent three additions per lane on the tree: 256 blobs 5.16 -> 4.91 ms, 64
// blobs 1.37 -> 1.25 ms, and with the shares fitted to the batch 21 blobs 1.20
// -> 0.42 ms, 9 blobs 0.38 -> 0.22 ms, 1 blob 0.19 -> 0.11 ms (the sums over more
// shares cost 0.05 to 0.07 ms of that at 1 to 64 blobs).  What bounds it at 256
// blobs is the multiply-adds: against a table cut to a few lines it takes 4.4
// ms, and the kernels after it get 7% faster too, so the gathers cost power
// more than time.
//
// The gathers come from a table far larger than any cache, and two waves per
// SIMD do not hide such a load behind each other's additions.  The lane runs
// one flat loop over its (term, window) pairs in two stages: the digit and the
// load of the next point are issued before the addition of the current one,
// and a term's scalar is loaded while the term before it is added (1 blob
// 0.228 -> 0.192 ms, 21 blobs 1.32 -> 1.20 ms).
//
// A wave takes items (share, 64 MSMs) from the counter q[0], cleared by the
// kernel that runs before, until the queue is drained, and leaves after one
// failed take; nj is a multiple of 64, so items are whole waves.
__global__ void __launch_bounds__(256, 2)
    k_phase_a(G1X *part, const Fr *scal, const G1AT *table, WindowPlan plan, uint32_t nj, uint32_t nblobs,
              uint32_t splits, uint32_t parts, uint32_t groups, uint32_t *q, uint32_t force_checked) {
    const uint32_t lane = threadIdx.x % 64;
    const uint32_t per_share = nblobs * splits * (nj / 64);  // items of 64 MSMs
    const uint32_t shares = parts * groups, nitems = per_share * shares;
    const uint32_t terms = 64 / parts;
#pragma unroll 1
    for (;;) {
        uint32_t item = 0;
        if (lane == 0) item = atomicAdd(q, 1u);
        item = __builtin_amdgcn_readfirstlane(item);
        if (item >= nitems) break;
        const uint32_t share = item / per_share;
        const uint32_t run = share / groups, g = share % groups;
        const uint32_t idx = (item % per_share) * 64 + lane;
        const uint32_t blob = idx % nblobs, js = idx / nblobs;
        const uint32_t j = js / splits, msm = (blob * splits + js % splits) * nj + j;
        const uint32_t w0 = g * plan.W / groups, w1 = (g + 1) * plan.W / groups;
        const Fr *sc = scal + (size_t)msm * 64 + run * terms;
        const G1AT *tab = table + (size_t)(j * 64 + run * terms) * plan.entries();
        G1X acc = g1x_identity();
        bool exc = force_checked != 0, started = false;
        if (w0 < w1) {  // (more groups than windows leave some empty)
            const uint32_t first = plan.bit(w0);
            uint32_t k = 0, w = w0;
            ScalarBits s;
            s.load(sc[0]);
            s.skip(first);
            Fr ahead = sc[terms > 1 ? 1 : 0];
            bool neg_next;
            uint32_t mag_next = window_digit(s.low(plan.c + plan.wide(w)), plan, w, s.neg, neg_next);
            G1A next = tab[plan.entry(w) + (mag_next ? mag_next - 1 : 0u)].p;
#pragma unroll 1
            for (;;) {
                const G1A pt = next;
                const bool neg = neg_next, skip = mag_next == 0;
                s.skip(plan.c + plan.wide(w));
                if (++w == w1) {
                    w = w0;
                    k++;
                    s.load(ahead);
                    s.skip(first);
                    if (k + 1 < terms) ahead = sc[k + 1];
                }
                const bool more = k < terms;
                if (more) {
                    mag_next = window_digit(s.low(plan.c + plan.wide(w)), plan, w, s.neg, neg_next);
                    next = tab[(size_t)k * plan.entries() + plan.entry(w) + (mag_next ? mag_next - 1 : 0u)].p;
                }
                if (!skip) {
                    if (started) {
                        acc = g1x_madd_acc(acc, pt, neg, exc);
                    } else {
                        acc = g1x_start(pt, neg, exc);
                        started = true;
                    }
                }
                if (!more) break;
            }
        }
        G1X *out = &part[(size_t)msm * shares + share];
        if (exc) phase_a_slow(out, sc, tab, plan, terms, w0, w1);
        else *out = acc;
    }
}

}  // namespace

hipError_t launch_phase_a(G1X *part, const Fr *scal, const G1AT *table, WindowPlan plan, uint32_t nj,
                          uint32_t nblobs, uint32_t splits, uint32_t parts, uint32_t groups, uint32_t grid, uint32_t *queue,
                          uint32_t force_checked, hipStream_t s) {
    if (parts == 0 || 64 % parts != 0 || nj % 64 != 0) return hipErrorInvalidValue;
    const uint32_t blocks = (nblobs * splits * (nj / 64) * parts * groups + 3) / 4;  // four waves each
    if (grid > blocks) grid = blocks;
    if (grid == 0) grid = 1;
    hipLaunchKernelGGL(k_phase_a, dim3(grid), dim3(256), 0, s, part, scal, table, plan, nj, nblobs, splits,
                       parts, groups, queue, force_checked);
    return hipGetLastError();
}

}  // namespace vkzg_amd
