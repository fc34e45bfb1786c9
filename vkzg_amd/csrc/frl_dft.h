// Transforms over Fr by single waves: DFT_64 of four columns and DFT_128 of two,
// 4 values per lane, in FrL (field_frl.h: 9 x 29-bit limbs, Montgomery radix
// 2^261, lazy sums) with FrL twiddle tables of 48-byte entries.  Used by the
// radix-4 recovery kernels and the FK20 scalars.
//
// They run as Stockham stages (natural order in and out): thread j of a column
// of length N reads d[j + r N / R] (r < R), multiplies by w_(Ns R)^((j mod Ns) r),
// takes the DFT_R and writes d'[(j / Ns) Ns R + j mod Ns + r Ns], for radices
// 4, 4, 4 (N = 64) and 4, 4, 4, 2 (N = 128), through a 256-value LDS region per
// wave.  Value bounds, in multiples of r, are noted where they matter.
#pragma once

#include "field_frl.h"

namespace vkzg_amd {

// Writes and reads of an exchange region by the lanes of one wave: the
// region is the wave's own, so a block-wide barrier (blocks of 1-4 waves)
// only has to order each wave's LDS accesses.
VKZG_DEV void exch_sync() { __syncthreads(); }

// A 48-byte FrL table entry (limbs 0-3, 4-7, 8 and padding).
VKZG_DEV FrL ld_frl_tab(const uint4 *tab, uint32_t k) {
    const uint4 *q = tab + 3u * k;
    const uint4 a = q[0], b = q[1];
    const uint32_t c = q[2].x;
    FrL r;
    r.v[0] = a.x, r.v[1] = a.y, r.v[2] = a.z, r.v[3] = a.w;
    r.v[4] = b.x, r.v[5] = b.y, r.v[6] = b.z, r.v[7] = b.w;
    r.v[8] = c;
    return r;
}
// Packed intermediates: 8 words per value.
VKZG_DEV FrL ld_frl(const Fr *p) {
    const uint4 *q = reinterpret_cast<const uint4 *>(p);
    const uint4 a = q[0], b = q[1];
    const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    return frl_unpack(w);
}
VKZG_DEV void st_frl(Fr *p, const FrL &v) {
    uint32_t w[8];
    frl_pack(w, v);
    uint4 *q = reinterpret_cast<uint4 *>(p);
    q[0] = make_uint4(w[0], w[1], w[2], w[3]);
    q[1] = make_uint4(w[4], w[5], w[6], w[7]);
}

// A wave's 256-value FrL exchange region (9 KiB): limbs 0-3 and 4-7 as two
// planes of 16-byte slots (bank-spread as Exch) and limb 8 as a plane of
// words.
struct Exch4 {
    uint4 *base;
    VKZG_DEV static uint32_t pos(uint32_t idx) { return idx ^ ((idx >> 5) & 7u); }
    VKZG_DEV void put(uint32_t idx, const FrL &v) const {
        const uint32_t p = pos(idx);
        base[p] = make_uint4(v.v[0], v.v[1], v.v[2], v.v[3]);
        base[256 + p] = make_uint4(v.v[4], v.v[5], v.v[6], v.v[7]);
        reinterpret_cast<uint32_t *>(base + 512)[p] = v.v[8];
    }
    VKZG_DEV FrL get(uint32_t idx) const {
        const uint32_t p = pos(idx);
        const uint4 a = base[p], b = base[256 + p];
        FrL r;
        r.v[0] = a.x, r.v[1] = a.y, r.v[2] = a.z, r.v[3] = a.w;
        r.v[4] = b.x, r.v[5] = b.y, r.v[6] = b.z, r.v[7] = b.w;
        r.v[8] = reinterpret_cast<const uint32_t *>(base + 512)[p];
        return r;
    }
};
constexpr uint32_t kExch4Uint4 = 576;  // 9 KiB per wave

// The transform's direction: tab[k] = w^k (FrL table), w4 = w^2048.
struct Dir4 {
    const uint4 *tab;
    FrL w4;
    VKZG_DEV explicit Dir4(const uint4 *t) : tab(t) { w4 = ld_frl_tab(tab, 2048); }
    VKZG_DEV FrL pow(uint32_t k) const { return ld_frl_tab(tab, k & 8191u); }
};

// out[e] = sum_b v[b] w4^(b e) (natural order in and out).  In: v0
// normalised (< V r), v1..v3 normalised below 2r.  Out: limbs below
// 3 * 2^30, values below (V + 10) r.  One product.
VKZG_DEV void dft4(FrL &v0, FrL &v1, FrL &v2, FrL &v3, const FrL &w4) {
    const FrL a = frl_add(v0, v2), b = frl_sub4(v0, v2);  // < V+2, < V+4
    const FrL c = frl_add(v1, v3), d = frl_sub4(v1, v3);  // < 4 (limbs < 2^30), < 6
    const FrL tw = frl_mul(d, w4);                        // < 2
    v0 = frl_add(a, c);                                   // < V+6
    v2 = frl_sub8(a, c);                                  // < V+10
    v1 = frl_add(b, tw);                                  // < V+6
    v3 = frl_sub4(b, tw);                                 // < V+8
}

// One radix-4 Stockham stage of a column at LDS offset `col` (length N,
// N / 4 threads, thread j): v <- d[j + r N/4] twiddled and transformed; the
// caller stores v at (j / Ns) 4 Ns + j mod Ns + r Ns.  v[0] is carried
// untwiddled, so it is normalised first; the twiddle products take v[1..3]
// back below 2r.
template <int N, int NS>
VKZG_DEV void stage4_load(FrL (&v)[4], const Dir4 &d, const Exch4 &x, uint32_t col, uint32_t j) {
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = x.get(col + j + (uint32_t)r * (N / 4));
    const uint32_t k = j % NS;
    v[0] = frl_norm(v[0]);
#pragma unroll
    for (int r = 1; r < 4; r++) v[r] = frl_mul(v[r], d.pow((8192u / (NS * 4)) * k * (uint32_t)r));
    dft4(v[0], v[1], v[2], v[3], d.w4);
}
template <int NS>
VKZG_DEV void stage4_store(const FrL (&v)[4], const Exch4 &x, uint32_t col, uint32_t j) {
    const uint32_t base = (j / NS) * NS * 4u + j % NS;
#pragma unroll
    for (int r = 0; r < 4; r++) x.put(col + base + (uint32_t)r * NS, v[r]);
}

// Pass B (DFT_64) of the wave's 4 columns cc (k2 = 2q + (cc & 1) + 64 (cc >> 1)):
// lane L = 4j + cc enters with v[r] = y[j + 16r][cc] (normalised, below 2r)
// and leaves with v[r] = X[j + 16r] of its column (below 32r).
VKZG_DEV void pass_b4(FrL (&v)[4], const Dir4 &d, const Exch4 &x, uint32_t lane) {
    const uint32_t cc = lane & 3u, j = lane >> 2, col = cc * 64u;
    dft4(v[0], v[1], v[2], v[3], d.w4);  // < 12
    exch_sync();
    stage4_store<1>(v, x, col, j);
    exch_sync();
    stage4_load<64, 4>(v, d, x, col, j);  // < 22
    exch_sync();
    stage4_store<4>(v, x, col, j);
    exch_sync();
    stage4_load<64, 16>(v, d, x, col, j);  // < 32; NS = 16: output index j + 16 r
}

// Pass A (DFT_128) of the wave's 2 columns c: lane L = 32c + j enters with
// v[r] = x[j + 32r] (normalised, below 2r) and leaves with the outputs
// k2 = pass_a4_k2(j, t).
VKZG_DEV uint32_t pass_a4_k2(uint32_t j, int t) {
    // t = 0, 1: j' = j, outputs j', j' + 64; t = 2, 3: j' = j + 32
    return j + 32u * (uint32_t)(t >> 1) + 64u * (uint32_t)(t & 1);
}
// The transform itself: v[t] at index pass_a4_k2(j, t), below 36r, limbs below
// 3 * 2^30 (a product's first operand).
VKZG_DEV void dft128(FrL (&v)[4], const Dir4 &d, const Exch4 &x, uint32_t lane) {
    const uint32_t c = lane >> 5, j = lane & 31u, col = c * 128u;
    dft4(v[0], v[1], v[2], v[3], d.w4);  // < 12
    exch_sync();
    stage4_store<1>(v, x, col, j);
    exch_sync();
    stage4_load<128, 4>(v, d, x, col, j);  // < 22
    exch_sync();
    stage4_store<4>(v, x, col, j);
    exch_sync();
    stage4_load<128, 16>(v, d, x, col, j);  // < 32
    exch_sync();
    stage4_store<16>(v, x, col, j);
    exch_sync();
    // radix-2 stage (Ns = 64): j' = j and j + 32, d[j'] and d[j' + 64],
    // twiddle w128^j' = w^(64 j')
    const FrL u0 = frl_norm(x.get(col + j)), u2 = frl_norm(x.get(col + j + 32u));
    const FrL t1 = frl_mul(x.get(col + j + 64u), d.pow(64u * j));           // < 2
    const FrL t3 = frl_mul(x.get(col + j + 96u), d.pow(64u * (j + 32u)));  // < 2
    v[0] = frl_add(u0, t1);   // < 34
    v[1] = frl_sub4(u0, t1);  // < 36
    v[2] = frl_add(u2, t3);
    v[3] = frl_sub4(u2, t3);
}
// The same with output v[t] multiplied by fac(t) (normalised, below 2r) instead
// of the four-step twiddle.
template <class F>
VKZG_DEV void pass_a4f(FrL (&v)[4], const Dir4 &d, const Exch4 &x, uint32_t lane, const F &fac) {
    dft128(v, d, x, lane);
#pragma unroll
    for (int t = 0; t < 4; t++) v[t] = frl_mul(v[t], fac(t));
}

}  // namespace vkzg_amd
