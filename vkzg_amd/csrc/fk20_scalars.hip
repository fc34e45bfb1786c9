// FK20 cell-proof kernels (the reference's computeBatch, src/vkzg.cpp:899-1039).
//
//   k_blob_dft       blob bytes -> canonical check -> first step of iNTT_4096
//   k_fk20_scalars   second step -> circulant columns -> NTT_128 -> phase-A
//                    scalars
//   k_phase_a        u[j] = sum_i scal[j][i] * xext[j][i]: fixed-base windowed
//                    MSM against the resident multiples table, a lane per share
//   k_sum_groups     the shares of each MSM summed
//   k_ladder         2^(8d) times the split-circulant folds of u
//   k_phase_b        phase-B buckets, one lane per (blob, output, bucket)
//   k_bucket_reduce  sum_k k * B[k-1] per output
//   k_finalize       C+ +- C-, affine, compressed, bit-reversed order

#include "frl_dft.h"
#include "ntt.h"
#include "proof_common.h"

namespace vkzg_amd {

namespace {
// The inverse transform of a blob's 4096 values as 64 x 64 (n = rho + 64 b,
// k = k1 + 64 k2):
//   c[rho + 64 b] = 1/4096 sum_k1 w64^-(b k1) [w^-(rho k1) sum_k2 p[k1 + 64 k2] w64^-(rho k2)]
// with w = omega_4096.  A circulant column takes the coefficients of one residue
// rho, so the second step's columns go straight into the circulant transforms.
// Waves of 4 columns each do both steps: 16 waves per blob for the first
// (k_blob_dft), 16 or 32 for the second.  A block per eight columns with the whole
// polynomial in its LDS, each repeating the whole inverse transform, spent 12
// block-wide stages on it: 142 us for a blob, 119 for 9, 255 for 256; two kernels of
// waves take 56, 50 and 157 us.
constexpr uint32_t kItems = 16;    // waves of four columns per blob
constexpr uint32_t kWaves = 4;     // waves per block

// Coefficient-step intermediates Y[k1][rho] of a blob in tiles of 4 rho x 4 k1
// (512 bytes), which a wave of either step writes or reads whole.
VKZG_DEV uint32_t y_index(uint32_t k1, uint32_t rho) {
    return ((rho >> 2) * kItems + (k1 >> 2)) * 16u + (rho & 3u) * 4u + (k1 & 3u);
}

// Item (blob, q): columns k1 = 4q + cc.  bad[item]: an element >= r in its columns.
// Clears the tile counter of the phase-A launch that follows.
__global__ void __launch_bounds__(64 * kWaves, 2)
    k_blob_dft(Fr *Y, uint32_t *bad, const uint8_t *blobs, uint64_t blob_stride, const uint4 *roots_inv,
               uint32_t *queue, uint32_t nitems) {
    __shared__ uint4 lds[kWaves * kExch4Uint4];
    if (blockIdx.x == 0 && threadIdx.x == 0) queue[0] = 0u;
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t item = blockIdx.x * kWaves + wave;
    if (item >= nitems) return;
    const uint32_t blob = item / kItems, q = item % kItems;
    const Exch4 x{lds + kExch4Uint4 * wave};
    const uint32_t cc = lane & 3u, j = lane >> 2, k1 = 4u * q + cc;
    // p[k1 + 64 k2] is element brev12(k1 + 64 k2) = 64 brev6(k1) + brev6(k2) of the
    // blob (k_blob_to_fr.comp:23-37), k2 = j + 16 r
    const uint32_t *src = reinterpret_cast<const uint32_t *>(blobs + blob_stride * blob) +
                          (64u * brev_bits(k1, 6) + 4u * brev_bits(j, 4)) * 8;
    const FrL conv = frl_const(cfrl::R2);
    bool over = false;
    FrL v[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        uint32_t w[8];
#pragma unroll
        for (int k = 0; k < 8; k++) w[k] = src[8u * brev_bits((uint32_t)r, 2) + k];
        const Fr e = fr_from_be_words(w);
        over |= !limbs_lt<8>(e.v, cfr::P);
        v[r] = frl_mul(frl_unpack(e.v), conv);  // any 256-bit value: below 3r
    }
    const uint64_t any = __ballot(over);
    if (lane == 0) bad[item] = any != 0;
    pass_b4(v, Dir4(roots_inv), x, lane);  // over k2: v[r] at rho = j + 16 r, < 32
    Fr *dst = Y + (size_t)blob * 4096;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const uint32_t rho = j + 16u * (uint32_t)r;
        st_frl(dst + y_index(k1, rho), frl_mul(v[r], ld_frl_tab(roots_inv, 2u * rho * k1)));
    }
}

// Item (blob, p, h): the circulant columns i = 63 - rho of rho = 4p + cc,
//   tc_i[0] = c[4095 - i], tc_i[128 - m] = c[4095 - i - 64 m] (m = 1..62), else 0,
// that is tc[0] = c_b at b = 63 and tc[t] at b = t - 65 (t = 66..127), and
// scal[j][i] = NTT_128(tc_i)[j] as sign and magnitude (k_build_circulant.comp:30-72),
// two columns at a time; `halves` = 2: one pair per wave (both waves of a pair
// repeat the DFT_64: half the chain, for batches that leave SIMDs idle).
// Segment m of a split ladder starts at 2^(kDigitBits lad_start(M, m)) u: its scalar
// set is the same values times that power of two.  The product that takes a
// transform's output out of Montgomery form takes the power along.
__global__ void __launch_bounds__(64 * kWaves, 2)
    k_fk20_scalars(Fr *scal, uint32_t *err, Fr *coeffs, const Fr *Y, const uint32_t *bad, const uint4 *roots,
                   const uint4 *roots_inv, uint32_t splits, uint32_t halves, Fr bias, uint32_t nitems) {
    __shared__ uint4 lds[kWaves * kExch4Uint4];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t item = blockIdx.x * kWaves + wave;
    if (item >= nitems) return;
    const uint32_t blob = item / (kItems * halves), p = item / halves % kItems, h0 = item % halves;
    const Exch4 x{lds + kExch4Uint4 * wave};
    const uint32_t cc = lane & 3u, jb = lane >> 2;
    FrL y[4];
#pragma unroll
    for (int r = 0; r < 4; r++) y[r] = ld_frl(Y + (size_t)blob * 4096 + y_index(jb + 16u * (uint32_t)r, 4u * p + cc));
    if (p == 0 && h0 == 0) {
        const uint64_t any = __ballot(lane < kItems && bad[blob * kItems + lane % kItems] != 0);
        if (lane == 0) err[blob] = any != 0;
    }
    pass_b4(y, Dir4(roots_inv), x, lane);  // over k1: y[r] at b = jb + 16 r
    const FrL inv_n = frl_const(cfrl::INV_4096_M);
#pragma unroll
    for (int r = 0; r < 4; r++) y[r] = frl_mul(y[r], inv_n);
    // Optionally the monomial coefficients, zero-padded to 8192, for the cell
    // extension (compute_cells_and_kzg_proofs).
    if (coeffs && h0 == 0) {
        Fr *cdst = coeffs + (size_t)blob * 8192;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const uint32_t n = 4u * p + cc + 64u * (jb + 16u * (uint32_t)r);
            Fr e;
            frl_pack(e.v, frl_mul(y[r], frl_const(cfrl::TO_R256)));
            fr_reduce_once(e.v, e.v);
            cdst[n] = e;
            cdst[n + 4096] = fr_zero();
        }
    }
    const Dir4 fwd(roots);
    const uint32_t c = lane >> 5, j = lane & 31u;
#pragma unroll 1
    for (uint32_t h = h0; h < 2; h += halves) {
        exch_sync();
#pragma unroll
        for (int r = 0; r < 4; r++) x.put(cc * 64u + jb + 16u * (uint32_t)r, y[r]);
        exch_sync();
        // tc[j + 32 r]
        const uint32_t col = (2u * h + c) * 64u;
        FrL v[4];
        v[0] = x.get(col + 63u);
        v[2] = x.get(col + (j > 0 ? j - 1u : 0u));
        v[3] = x.get(col + 31u + j);
#pragma unroll
        for (int k = 0; k < 9; k++) {
            v[0].v[k] = j == 0 ? v[0].v[k] : 0u;
            v[1].v[k] = 0u;
            v[2].v[k] = j >= 2 ? v[2].v[k] : 0u;
        }
        dft128(v, fwd, x, lane);
        Fr *out = scal + (size_t)blob * splits * 8192 + (63u - 4u * p - 2u * h - c);
#pragma unroll 1
        for (uint32_t m = 0; m < splits; m++) {
            const uint32_t bit = kDigitBits * lad_start(splits, m);
            FrL power;
#pragma unroll
            for (uint32_t k = 0; k < 9; k++) power.v[k] = bit / 29 == k ? 1u << (bit % 29) : 0u;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                Fr e;
                frl_pack(e.v, frl_mul(v[t], power));
                fr_reduce_once(e.v, e.v);
                out[(size_t)m * 8192 + pass_a4_k2(j, t) * 64u] = biased_magnitude(e, bias);
            }
        }
    }
}

}  // namespace

hipError_t launch_fk20_scalars(Fr *scal, const uint8_t *blobs, uint64_t blob_stride, uint32_t *err, void *scratch,
                               const uint4 *roots, const uint4 *roots_inv, uint32_t *queue, Fr *coeffs,
                               uint32_t splits, uint32_t nblobs, uint32_t cus, WindowPlan plan, hipStream_t s) {
    Fr *Y = static_cast<Fr *>(scratch);
    uint32_t *bad = reinterpret_cast<uint32_t *>(Y + (size_t)nblobs * 4096);
    const uint32_t n1 = nblobs * kItems;
    hipLaunchKernelGGL(k_blob_dft, dim3(blocks_for(n1, kWaves)), dim3(64 * kWaves), 0, s, Y, bad, blobs, blob_stride,
                       roots_inv, queue, n1);
    // two waves per four columns while they are at most one per SIMD
    const uint32_t halves = (uint64_t)n1 * 2 <= (uint64_t)cus * 4 ? 2 : 1, n2 = n1 * halves;
    hipLaunchKernelGGL(k_fk20_scalars, dim3(blocks_for(n2, kWaves)), dim3(64 * kWaves), 0, s, scal, err, coeffs, Y, bad,
                       roots, roots_inv, splits, halves, scalar_bias(plan), n2);
    return hipGetLastError();
}

}  // namespace vkzg_amd
