// Variable-base multi-scalar multiplication on G1 (Pippenger's bucket method
// with the GLV split), for the sums of batch cell-proof verification (for
// commitments, over fixed points, phase A's kernel and a multiples table).  No
// reference counterpart: the reference only has the FK20
// MSMs with fixed scalars or fixed points (k_phase_a.comp, k_phase_b_split.comp).
//
// Several independent sums ("MSMs") run in one launch sequence.  Entry e adds
// [scalar_e] P_{pidx_e} to MSM mid_e.  Each scalar is split k = k1 + LAMBDA k2
// (glv.h), so entry e becomes two half-entries: (P, k1) and (phi(P), k2) with
// 128-bit scalars.  Then, for windows of c bits and signed digits in
// [-2^(c-1), 2^(c-1)]:
//   count    histogram of (msm, window, |digit|) keys     (atomics)
//   scan     bucket offsets (one block; three passes above 16k buckets)
//   scatter  point references sorted by key               (atomics)
//   buckets  one lane (XYZZ, checked) or four quads (homogeneous) per bucket
//            sum its points; buckets of more than 24 points by a wave
//   windows  blocks per (msm, window): sum_b (b+1) B_b by running sums over
//            segments of at most 4 buckets on quads, then trees in LDS
//   combine  a wave per MSM: Horner over runs of windows (c doublings each) on
//            its quads, a tree, and the conversion to affine.
// The point order inside a bucket depends on atomics, but the sum is the same
// group element, so results are deterministic after normalisation.
#include "msm.h"

#include "proj_quad.h"

#include "glv.h"
#include "proof_common.h"

namespace vkzg_amd {

namespace {

constexpr uint32_t kWinQuads = 64;
constexpr uint32_t kHotLen = 24;    // longer buckets are summed by a wave (k_msm_hot)
constexpr uint32_t kWinSeg = 4;     // buckets per window quad: the sums are latency-bound
constexpr uint32_t kHotBlocks = 2048;
constexpr uint32_t kScanOneBlock = 16384;  // larger scans use k_msm_scan_tiles
constexpr uint32_t kScanTile = 4096;       // buckets per block of k_msm_scan_tiles
constexpr uint32_t kPtMask = (1u << 30) - 1;

// Signed digit w of a 128-bit scalar (4 words) with window c; carry in/out.
VKZG_DEV int32_t digit_at(const uint32_t *s, uint32_t w, uint32_t c, uint32_t &carry) {
    const uint32_t bit = w * c;
    uint32_t v = 0;
    if (bit < 128) {
        const uint32_t wi = bit >> 5, sh = bit & 31u;
        uint64_t x = s[wi];
        if (wi + 1 < 4) x |= (uint64_t)s[wi + 1] << 32;
        v = (uint32_t)(x >> sh) & ((1u << c) - 1u);
    }
    v += carry;
    const uint32_t half = 1u << (c - 1);
    if (v > half) {
        carry = 1;
        return (int32_t)v - (int32_t)(1u << c);
    }
    carry = 0;
    return (int32_t)v;
}

__global__ void k_msm_split(uint32_t *hs, const Fr *sc, uint32_t ne) {
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ne) return;
    uint32_t k1[4], k2[4];
    glv::split(k1, k2, sc[e].v);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        hs[8 * e + i] = k1[i];
        hs[8 * e + 4 + i] = k2[i];
    }
}

__global__ void k_msm_zero(uint32_t *a, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0;
}

__global__ void k_msm_count(uint32_t *cnt, const uint32_t *hs, const uint8_t *mid, uint32_t nh, uint32_t c,
                            uint32_t W) {
    const uint32_t h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= nh) return;
    const uint32_t *s = hs + 4 * h;
    const uint32_t base = (uint32_t)mid[h >> 1] * W;
    const uint32_t bk = 1u << (c - 1);
    uint32_t carry = 0;
#pragma unroll 1
    for (uint32_t w = 0; w < W; w++) {
        const int32_t d = digit_at(s, w, c, carry);
        if (d != 0) atomicAdd(&cnt[(base + w) * bk + (uint32_t)(d < 0 ? -d : d) - 1], 1u);
    }
}

// Exclusive scan of cnt[0..K) into off[0..K] (one block of 1024 threads);
// cur = off (the scatter cursors).
__global__ void __launch_bounds__(1024) k_msm_scan(uint32_t *off, uint32_t *cur, const uint32_t *cnt,
                                                   uint32_t K) {
    __shared__ uint32_t part[1024];
    const uint32_t t = threadIdx.x;
    const uint32_t per = (K + 1023) / 1024;
    const uint32_t lo = t * per, hi = lo + per < K ? lo + per : K;
    uint32_t sum = 0;
    for (uint32_t k = lo; k < hi; k++) sum += cnt[k];
    part[t] = sum;
    __syncthreads();
    for (uint32_t d = 1; d < 1024; d <<= 1) {
        const uint32_t v = t >= d ? part[t - d] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    uint32_t run = part[t] - sum;  // exclusive prefix of this thread's range
    for (uint32_t k = lo; k < hi; k++) {
        off[k] = run;
        cur[k] = run;
        run += cnt[k];
    }
    if (t == 1023) off[K] = part[1023];
}

// Three-pass form for large K.  Pass 1: each block scans its tile of
// kScanTile counts (4 per thread) into tile-local exclusive offsets and
// writes the tile total.
__global__ void __launch_bounds__(1024) k_msm_scan_tiles(uint32_t *off, uint32_t *tot, const uint32_t *cnt,
                                                         uint32_t K) {
    __shared__ uint32_t part[1024];
    const uint32_t t = threadIdx.x;
    const uint32_t lo = blockIdx.x * kScanTile + 4 * t;
    uint32_t v[4], sum = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v[i] = lo + i < K ? cnt[lo + i] : 0;
        sum += v[i];
    }
    part[t] = sum;
    __syncthreads();
    for (uint32_t d = 1; d < 1024; d <<= 1) {
        const uint32_t x = t >= d ? part[t - d] : 0;
        __syncthreads();
        part[t] += x;
        __syncthreads();
    }
    uint32_t run = part[t] - sum;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (lo + i < K) off[lo + i] = run;
        run += v[i];
    }
    if (t == 1023) tot[blockIdx.x] = part[1023];
}

// Pass 2 (one block): exclusive scan of the ntiles <= 1024 tile totals in
// place; off[K] = the grand total.
__global__ void __launch_bounds__(1024) k_msm_scan_totals(uint32_t *off, uint32_t *tot, uint32_t ntiles,
                                                          uint32_t K) {
    __shared__ uint32_t part[1024];
    const uint32_t t = threadIdx.x;
    const uint32_t mine = t < ntiles ? tot[t] : 0;
    part[t] = mine;
    __syncthreads();
    for (uint32_t d = 1; d < 1024; d <<= 1) {
        const uint32_t x = t >= d ? part[t - d] : 0;
        __syncthreads();
        part[t] += x;
        __syncthreads();
    }
    if (t < ntiles) tot[t] = part[t] - mine;
    if (t == 1023) off[K] = part[1023];
}

// Pass 3: add each tile's offset; cur = off.
__global__ void k_msm_scan_add(uint32_t *off, uint32_t *cur, const uint32_t *tot, uint32_t K) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= K) return;
    const uint32_t o = off[k] + tot[k / kScanTile];
    off[k] = o;
    cur[k] = o;
}

__global__ void k_msm_scatter(uint32_t *list, uint32_t *cur, const uint32_t *hs, const uint8_t *mid,
                              const uint32_t *pidx, uint32_t nh, uint32_t c, uint32_t W) {
    const uint32_t h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= nh) return;
    const uint32_t *s = hs + 4 * h;
    const uint32_t base = (uint32_t)mid[h >> 1] * W;
    const uint32_t bk = 1u << (c - 1);
    const uint32_t ref = pidx[h >> 1] | ((h & 1u) << 30);
    uint32_t carry = 0;
#pragma unroll 1
    for (uint32_t w = 0; w < W; w++) {
        const int32_t d = digit_at(s, w, c, carry);
        if (d == 0) continue;
        const uint32_t key = (base + w) * bk + (uint32_t)(d < 0 ? -d : d) - 1;
        const uint32_t pos = atomicAdd(&cur[key], 1u);
        list[pos] = ref | (d < 0 ? 0x80000000u : 0u);
    }
}

// The point a sorted reference names: phi(P) when bit 30 is set, negated when bit 31 is.
VKZG_DEV G1A msm_point(const G1A *pts, uint32_t ref) {
    G1A p = pts[ref & kPtMask];
    if (ref & (1u << 30)) p.x = fp_mul(p.x, fp_const(cfp::BETA_M));
    return g1a_neg_if(p, (ref >> 31) != 0);
}

// A bucket summed with the checked addition (a doubling or cancellation
// inside it, flagged by the call-free loop of k_msm_buckets).
VKZG_DEV_COLD void bucket_checked(G1X *acc, const G1A *pts, const uint32_t *list, uint32_t lo, uint32_t hi) {
    G1X a = g1x_identity();
    for (uint32_t q = lo; q < hi; q++) a = g1x_madd(a, msm_point(pts, list[q]));
    *acc = a;
}

// One lane per bucket (launches that fill the chip so).  A bucket with more than
// kHotLen points (the few digits of a narrow top window collect most points of
// every scalar) goes to the hot list instead, for k_msm_hot.
__global__ void __launch_bounds__(64) k_msm_buckets(G1P *buckets, const uint32_t *off, const uint32_t *list, const G1A *pts,
                              uint32_t K, uint32_t *hot, uint32_t *hot_n) {
    const uint32_t key = blockIdx.x * blockDim.x + threadIdx.x;
    if (key >= K) return;
    const uint32_t lo = off[key], hi = off[key + 1];
    if (hi - lo > kHotLen) {
        hot[atomicAdd(hot_n, 1u)] = key;
        return;
    }
    G1X acc = g1x_identity();
    bool exc = false;
#pragma unroll 1
    for (uint32_t q = lo; q < hi; q++) acc = g1x_madd_fast(acc, msm_point(pts, list[q]), exc);
    if (exc) bucket_checked(&acc, pts, list, lo, hi);
    buckets[key] = g1p_from_xyzz_lane(acc);
}

// msm_point in homogeneous coordinates
VKZG_DEV G1P msm_point_homog(const G1A *pts, uint32_t ref) {
    const G1A p = pts[ref & kPtMask];
    const Fp nu = fp_select((ref & (1u << 30)) != 0, fp_const(cfp::NU_BETA_M), fp_const(cfp::NU_M));
    const bool inf = g1a_is_identity(p);
    return G1P{fp_mul(p.x, nu), fp_select(inf, fp_one(), fp_cond_neg(p.y, (ref >> 31) != 0)),
               fp_select(inf, fp_zero(), fp_const(cfp::SIGMA_M))};
}

// The points list[lo..hi) summed by QUADS consecutive quads of one wave (quad k of
// them: every QUADS-th point, then a tree): complete additions in homogeneous
// coordinates (proj_quad.h), 3.5 rounds of products and one for a point's x.
template <uint32_t QUADS>
VKZG_DEV G1PQ quads_sum(const G1A *pts, const uint32_t *list, uint32_t lo, uint32_t hi, uint32_t k, uint32_t q) {
    G1PQ acc = g1p_spread(g1p_identity(), q);
#pragma unroll 1
    for (uint32_t i = lo + k; i < hi; i += QUADS) {
        const G1P p = msm_point_homog(pts, list[i]);
        acc = i == lo + k ? g1p_spread(p, q) : g1p_add_quad(g1p_gather(acc), p, q);
    }
#pragma unroll 1
    for (uint32_t m = 1; m < QUADS; m <<= 1) {
        const G1PQ other = g1pq_shfl_xor(acc, (int)(4 * m));
        acc = g1p_add_quad(g1p_gather(acc), g1p_gather(other), q);
    }
    return acc;
}
VKZG_DEV void g1pq_store(G1P *out, const G1PQ &p, uint32_t q) {
    const Fp y = g1pq_y(p);
    if (q == 0) out->y = y;
    else if (q == 2) out->x = p.r;
    else if (q == 3) out->z = p.r;
}

// Four quads per bucket, for launches that leave SIMDs idle with a lane each: there
// a bucket's chain of up to kHotLen additions is the time (a check of 128 cells:
// 170 -> 37 us).
__global__ void __launch_bounds__(64) k_msm_buckets_quads(G1P *buckets, const uint32_t *off, const uint32_t *list,
                                                          const G1A *pts, uint32_t K, uint32_t *hot, uint32_t *hot_n) {
    const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t key = tid / 16, k = (tid >> 2) & 3u, q = tid & 3u;
    if (key >= K) return;
    const uint32_t lo = off[key], hi = off[key + 1];
    if (hi - lo > kHotLen) {
        if ((tid & 15u) == 0) hot[atomicAdd(hot_n, 1u)] = key;
        return;
    }
    const G1PQ acc = quads_sum<4>(pts, list, lo, hi, k, q);
    if (k == 0) g1pq_store(&buckets[key], acc, q);
}

// Hot buckets, one wave (16 quads) each; blocks stride over the list.  A check of
// 128 cells: 135 -> 74 us against a lane per share and a tree of lanes.
__global__ void __launch_bounds__(64) k_msm_hot(G1P *buckets, const uint32_t *off, const uint32_t *list,
                                                const G1A *pts, const uint32_t *hot, const uint32_t *hot_n) {
    const uint32_t k = threadIdx.x >> 2, q = threadIdx.x & 3u;
    const uint32_t n = *hot_n;
#pragma unroll 1
    for (uint32_t h = blockIdx.x; h < n; h += gridDim.x) {
        const uint32_t key = hot[h];
        const G1PQ acc = quads_sum<16>(pts, list, off[key], off[key + 1], k, q);
        if (k == 0) g1pq_store(&buckets[key], acc, q);
    }
}

// [k] p, 0 < k < 2^16, by a quad
VKZG_DEV G1PQ g1p_mul_small(const G1P &p, uint32_t k, uint32_t q) {
    G1PQ acc = g1p_spread(p, q);
#pragma unroll 1
    for (int b = 30 - __builtin_clz(k); b >= 0; b--) {
        acc = g1pq_dbl(acc, q);
        if ((k >> b) & 1u) acc = g1p_add_quad(g1p_gather(acc), p, q);
    }
    return acc;
}

// The sum of the block's kWinQuads points, one per quad, in its quad 0.
VKZG_DEV G1PQ g1pq_block_sum(G1PQ acc, Fp *sh, uint32_t t) {
#pragma unroll 1
    for (uint32_t stride = kWinQuads / 2; stride > 0; stride >>= 1) {
        __syncthreads();
        sh[t] = acc.r;
        __syncthreads();
        if (t / 4 < stride)
            acc = g1p_add_quad(g1p_gather(acc), g1p_gather(G1PQ{sh[t + 4 * stride]}), t & 3u);
    }
    return acc;
}
// Block (msm, window, part): sum over the part's buckets b of (b + 1) B_b.
// Quad k owns buckets [lo, lo + seg): running sums from the top give R = sum B_b
// and T = sum (b - lo + 1) B_b, and its share is T + lo R; a tree adds the
// shares.  A window's parts (enough of them for at most kWinSeg buckets per
// quad) are added by k_msm_parts.  The chain of additions and doublings is the
// time here, so quads in homogeneous coordinates run it (proj_quad.h): with 38
// windows of 64 buckets (the sums of a check of 128 cells) 285 -> 76 us against
// a lane per bucket in XYZZ coordinates.
__global__ void __launch_bounds__(4 * kWinQuads) k_msm_windows(G1P *wpart, const G1P *buckets, uint32_t bk,
                                                               uint32_t parts) {
    __shared__ Fp sh[4 * kWinQuads];
    const uint32_t t = threadIdx.x, q = t & 3u, k = t >> 2;
    const uint32_t win = blockIdx.x / parts, part = blockIdx.x % parts;
    const G1P *B = buckets + (size_t)win * bk;
    const uint32_t per_part = bk / parts;
    const uint32_t seg = per_part > kWinQuads ? per_part / kWinQuads : 1;
    const uint32_t lo = part * per_part + k * seg;
    G1PQ share = g1p_spread(g1p_identity(), q);
    if (k * seg < per_part) {
        G1P R = B[lo + seg - 1];
        if (seg == 1) {
            share = g1p_mul_small(R, lo + 1, q);
        } else {
            G1P T = R;
#pragma unroll 1
            for (uint32_t b = lo + seg - 1; b-- > lo;) {
                R = g1p_gather(g1p_add_quad(R, B[b], q));
                T = g1p_gather(g1p_add_quad(T, R, q));
            }
            share = lo ? g1p_add_quad(g1p_gather(g1p_mul_small(R, lo, q)), T, q) : g1p_spread(T, q);
        }
    }
    share = g1pq_block_sum(share, sh, t);
    if (k == 0) g1pq_store(&wpart[blockIdx.x], share, q);
}

// wsum[win] = sum of the window's parts (at most kWinQuads of them).
__global__ void __launch_bounds__(4 * kWinQuads) k_msm_parts(G1P *wsum, const G1P *wpart, uint32_t parts) {
    __shared__ Fp sh[4 * kWinQuads];
    const uint32_t t = threadIdx.x, q = t & 3u, k = t >> 2;
    const G1P p = k < parts ? wpart[(size_t)blockIdx.x * parts + k] : g1p_identity();
    const G1PQ acc = g1pq_block_sum(g1p_spread(p, q), sh, t);
    if (k == 0) g1pq_store(&wsum[blockIdx.x], acc, q);
}

// out[m] = sum_w 2^(c w) wsum[m W + w], affine ((0, 0) for the identity), by
// wave m.  The chain of c (W - 1) doublings is this launch's critical path, so
// it runs on quads in homogeneous coordinates (two rounds of products per
// doubling, complete additions: proj_quad.h).  The additions would lengthen it
// by 3.5 rounds each, so the wave's 16 quads each take a run of L = ceil(W / 16)
// windows, from the top down, by Horner, double their sum up to its place and
// meet in a tree: L + 3 additions in the chain instead of W - 1.  With 19 windows
// of 7 bits (the sums of a check of 128 cells), 730 us for a quad's three-round
// XYZZ Horner -> 410 us.
__global__ void __launch_bounds__(64) k_msm_combine(G1A *out, const G1P *wsum, uint32_t W, uint32_t c) {
    const uint32_t m = blockIdx.x, g = threadIdx.x >> 2, q = threadIdx.x & 3u;
    const G1P *ws = wsum + (size_t)m * W;
    const uint32_t L = (W + 15) / 16;
    const uint32_t hi = W > g * L ? W - g * L : 0, lo = hi > L ? hi - L : 0;
    G1P acc = hi > 0 ? ws[hi - 1] : g1p_identity();
    G1PQ a = g1p_spread(acc, q);
#pragma unroll 1
    for (uint32_t w = hi; w > lo + 1;) {
        w--;
#pragma unroll 1
        for (uint32_t i = 0; i < c; i++) a = g1pq_dbl(a, q);
        a = g1p_add_quad(g1p_gather(a), ws[w - 1], q);
    }
    // the wave runs as long as its longest chain: quad 0's, c (W - 1) in all
#pragma unroll 1
    for (uint32_t i = 0; i < lo * c; i++) a = g1pq_dbl(a, q);
#pragma unroll 1
    for (uint32_t x = 4; x < 64; x <<= 1) {
        G1PQ b;
#pragma unroll
        for (int i = 0; i < kFpLimbs; i++) b.r.v[i] = __shfl_xor(a.r.v[i], (int)x);
        a = g1p_add_quad(g1p_gather(a), g1p_gather(b), q);
    }
    acc = g1p_gather(a);
    G1A r = g1a_identity();
    if (!fp_is_zero(acc.z)) {
        const Fp inv = fp_inv(acc.z);
        r.x = fp_mul(fp_mul(acc.x, fp_const(cfp::SIGMA_OVER_NU_M)), inv);
        r.y = fp_mul(fp_mul(acc.y, fp_const(cfp::SIGMA_M)), inv);
    }
    if (threadIdx.x == 0) out[m] = r;
}

}  // namespace

MsmShape msm_shape(uint32_t ne, uint32_t nmsm) {
    MsmShape sh;
    sh.ne = ne;
    sh.nmsm = nmsm;
    // about four half-entries per bucket and window: 2^(c-1) ~ per / 4
    const uint32_t per = nmsm ? (2 * ne + nmsm - 1) / nmsm : 0;
    uint32_t c = 4;
    while (c < 13 && (1u << (c + 2)) <= per) c++;
    sh.c = c;
    sh.W = (129 + c - 1) / c;
    sh.bk = 1u << (c - 1);
    sh.K = nmsm * sh.W * sh.bk;
    sh.parts = sh.bk > kWinQuads * kWinSeg ? sh.bk / (kWinQuads * kWinSeg) : 1;
    return sh;
}

size_t msm_scratch_bytes(const MsmShape &sh) {
    const size_t nh = 2ull * sh.ne;
    size_t b = 0;
    b += 16 * nh;                        // half scalars
    b += 4ull * (4 * (size_t)sh.K + 3);  // cnt (+ hot count), cur, off, hot list
    b += 4ull * (sh.K / kScanTile + 1);  // scan tile totals
    b += 4 * nh * sh.W;                  // sorted references
    b += sizeof(G1P) * (size_t)sh.K;     // buckets
    b += sizeof(G1P) * (size_t)sh.nmsm * sh.W * (sh.parts + 1);
    return b + 16 * 256;  // each of the 10 regions is rounded up to 256 bytes
}

hipError_t launch_msm(const MsmShape &sh, void *scratch, const G1A *pts, const uint32_t *pidx, const Fr *sc,
                      const uint8_t *mid, G1A *out, uint32_t cus, hipStream_t s) {
    if (sh.ne == 0 || sh.nmsm == 0) return hipErrorInvalidValue;
    const uint32_t nh = 2 * sh.ne;
    uint8_t *p = static_cast<uint8_t *>(scratch);
    auto take = [&p](size_t bytes) {
        uint8_t *r = p;
        p += (bytes + 255) & ~size_t(255);
        return r;
    };
    uint32_t *hs = reinterpret_cast<uint32_t *>(take(16ull * nh));
    uint32_t *cnt = reinterpret_cast<uint32_t *>(take(4ull * (sh.K + 1)));  // cnt[K]: hot-bucket count
    uint32_t *hot = reinterpret_cast<uint32_t *>(take(4ull * sh.K));
    uint32_t *cur = reinterpret_cast<uint32_t *>(take(4ull * sh.K));
    uint32_t *off = reinterpret_cast<uint32_t *>(take(4ull * (sh.K + 1)));
    const uint32_t ntiles = (sh.K + kScanTile - 1) / kScanTile;
    uint32_t *tot = reinterpret_cast<uint32_t *>(take(4ull * (sh.K / kScanTile + 1)));
    uint32_t *list = reinterpret_cast<uint32_t *>(take(4ull * nh * sh.W));
    G1P *buckets = reinterpret_cast<G1P *>(take(sizeof(G1P) * (size_t)sh.K));
    G1P *wpart = reinterpret_cast<G1P *>(take(sizeof(G1P) * (size_t)sh.nmsm * sh.W * sh.parts));
    G1P *wsum = sh.parts > 1 ? reinterpret_cast<G1P *>(take(sizeof(G1P) * (size_t)sh.nmsm * sh.W)) : wpart;
    if ((size_t)(p - static_cast<uint8_t *>(scratch)) > msm_scratch_bytes(sh)) return hipErrorInvalidValue;
    if (sh.K > kScanOneBlock && ntiles > 1024) return hipErrorInvalidValue;  // beyond 4M buckets
    hipLaunchKernelGGL(k_msm_split, dim3(blocks_for(sh.ne, 256)), dim3(256), 0, s, hs, sc, sh.ne);
    hipLaunchKernelGGL(k_msm_zero, dim3(blocks_for(sh.K + 1, 256)), dim3(256), 0, s, cnt, sh.K + 1);
    hipLaunchKernelGGL(k_msm_count, dim3(blocks_for(nh, 256)), dim3(256), 0, s, cnt, hs, mid, nh, sh.c, sh.W);
    if (sh.K <= kScanOneBlock) {
        hipLaunchKernelGGL(k_msm_scan, dim3(1), dim3(1024), 0, s, off, cur, cnt, sh.K);
    } else {
        hipLaunchKernelGGL(k_msm_scan_tiles, dim3(ntiles), dim3(1024), 0, s, off, tot, cnt, sh.K);
        hipLaunchKernelGGL(k_msm_scan_totals, dim3(1), dim3(1024), 0, s, off, tot, ntiles, sh.K);
        hipLaunchKernelGGL(k_msm_scan_add, dim3(blocks_for(sh.K, 256)), dim3(256), 0, s, off, cur, tot, sh.K);
    }
    hipLaunchKernelGGL(k_msm_scatter, dim3(blocks_for(nh, 256)), dim3(256), 0, s, list, cur, hs, mid, pidx, nh,
                       sh.c, sh.W);
    // four quads per bucket while they are at most one wave per SIMD
    if (sh.K * 16ull <= (uint64_t)cus * 4 * 64)
        hipLaunchKernelGGL(k_msm_buckets_quads, dim3(blocks_for(sh.K * 16ull, 64)), dim3(64), 0, s, buckets, off, list,
                           pts, sh.K, hot, cnt + sh.K);
    else
        hipLaunchKernelGGL(k_msm_buckets, dim3(blocks_for(sh.K, 64)), dim3(64), 0, s, buckets, off, list, pts, sh.K,
                           hot, cnt + sh.K);
    const dim3 hot_grid(sh.K < kHotBlocks ? sh.K : kHotBlocks);
    hipLaunchKernelGGL(k_msm_hot, hot_grid, dim3(64), 0, s, buckets, off, list, pts, hot, cnt + sh.K);
    hipLaunchKernelGGL(k_msm_windows, dim3(sh.nmsm * sh.W * sh.parts), dim3(4 * kWinQuads), 0, s, wpart, buckets,
                       sh.bk, sh.parts);
    if (sh.parts > 1)
        hipLaunchKernelGGL(k_msm_parts, dim3(sh.nmsm * sh.W), dim3(4 * kWinQuads), 0, s, wsum, wpart, sh.parts);
    hipLaunchKernelGGL(k_msm_combine, dim3(sh.nmsm), dim3(64), 0, s, out, wsum, sh.W, sh.c);
    return hipGetLastError();
}

}  // namespace vkzg_amd
