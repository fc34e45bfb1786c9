// Helpers shared by the proof kernels.
#pragma once

#include "curve.h"
#include "kernels.h"
#include "ntt.h"

namespace vkzg_amd {

inline uint32_t blocks_for(uint64_t n, uint32_t bs) { return (uint32_t)((n + bs - 1) / bs); }

// The form phase A reads: sign (bit 255) and magnitude (below 2^254) plus the
// plan's digit bias.
VKZG_DEV Fr biased_magnitude(const Fr &canonical, const Fr &bias) {
    const Fr m = fr_signed_magnitude(canonical);
    Fr r;
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint64_t x = (uint64_t)m.v[i] + bias.v[i] + c;
        r.v[i] = (uint32_t)x;
        c = (uint32_t)(x >> 32);
    }
    return r;
}

// sum over the windows below the top one of (2^(width - 1) - 1) 2^bit: added
// to a magnitude below 2^254 it stays below 2^255, and each of those windows'
// bits then are its signed digit plus 2^(width - 1) - 1.
inline Fr scalar_bias(const WindowPlan &plan) {
    Fr r{};
    for (uint32_t w = 0; w + 1 < plan.W; w++) {
        const uint64_t v = (plan.H() << plan.wide(w)) - 1;
        const uint32_t li = plan.bit(w) >> 5;
        uint64_t c = v << (plan.bit(w) & 31u);
        for (uint32_t i = li; i < 8 && c; i++) {
            c += r.v[i];
            r.v[i] = (uint32_t)c;
            c >>= 32;
        }
    }
    return r;
}

VKZG_DEV G1X g1x_shfl_xor(const G1X &p, int m) {
    G1X o;
#pragma unroll
    for (int k = 0; k < kFpLimbs; k++) {
        o.x.v[k] = __shfl_xor(p.x.v[k], m);
        o.y.v[k] = __shfl_xor(p.y.v[k], m);
        o.zz.v[k] = __shfl_xor(p.zz.v[k], m);
        o.zzz.v[k] = __shfl_xor(p.zzz.v[k], m);
    }
    return o;
}

// The point lane (this lane + d) holds (lanes past the wave's end read their own).
VKZG_DEV G1X g1x_shfl_down(const G1X &p, uint32_t d) {
    G1X o;
#pragma unroll
    for (int k = 0; k < kFpLimbs; k++) {
        o.x.v[k] = __shfl_down(p.x.v[k], d);
        o.y.v[k] = __shfl_down(p.y.v[k], d);
        o.zz.v[k] = __shfl_down(p.zz.v[k], d);
        o.zzz.v[k] = __shfl_down(p.zzz.v[k], d);
    }
    return o;
}

}  // namespace vkzg_amd
