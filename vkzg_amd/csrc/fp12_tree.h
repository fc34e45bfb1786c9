// Exchanges between lanes and the sum over a group of 32 lanes that an Fp12
// product (tower.h) ends in.  Plain C++ apart from the exchange builtins, so
// tests/c builds it with g++ on 32 threads.
#pragma once

#include "field_fp.h"

namespace vkzg_amd {

VKZG_DEV Fp fp_shfl_xor(const Fp &v, int mask) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = __shfl_xor(v.v[i], mask);
    return r;
}

// DPP within rows of 16 lanes: lane l takes the value of lane l + n (kRowShl + n,
// lanes past the row's end 0) or l - n mod 16 (kRowRor + n).
constexpr int kRowShl = 0x100, kRowRor = 0x120;
template <int CTRL>
VKZG_DEV Fp fp_row_dpp(const Fp &v) {
    Fp r;
#pragma unroll
    for (int i = 0; i < kFpLimbs; i++) r.v[i] = __builtin_amdgcn_mov_dpp(v.v[i], CTRL, 0xf, 0xf, true);
    return r;
}

// The place of lane t's term in its group of 32 lanes: three terms in each row of
// 16, one per quad; the fourth quad's lanes (3 and 7 by quad) have none.
VKZG_DEV uint32_t fp12_term(uint32_t t) { return t % 32 / 16 * 3 + t % 16 / 4; }
VKZG_DEV bool fp12_has_term(uint32_t t) { return t % 16 < 12; }

// The sum of a group's six terms, in every lane by its place in the quad (zero
// where a lane has no term).  A term is the sum or difference of two products, so
// its limbs lie in [-2^30, 2^30) and two just fit 32 bits: the rows are added
// first, under one carry pass, which leaves at most 2^29 + 2, and then the three
// sums of a row, below 3 (2^29 + 2) < 2^31, by two rotations (the fourth quad's
// zero makes them whole in every quad), with a carry pass at the end.  Adding
// within the rows first would leave four normalised sums for the last pass, which
// can pass 2^31.
VKZG_DEV Fp fp12_tree(Fp v) {
    v = fp_norm_wide(fp_add_raw(v, fp_shfl_xor(v, 16)));
    v = fp_add_raw(v, fp_row_dpp<kRowRor + 4>(v));
    return fp_norm_wide(fp_add_raw(v, fp_row_dpp<kRowRor + 8>(v)));
}

}  // namespace vkzg_amd
