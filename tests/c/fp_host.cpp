// Host build of vkzg_amd/csrc/field_fp.h for tests/test_fp_model.py.  Reads
// lines "op k a.. b.. c.. d.." (13 signed limbs each), prints the 13 limbs of
// the result.  Built with -ftrapv, so a column that overflows its signed
// 64-bit accumulator (or a limb its 32 bits) aborts.
#define __host__
#define __device__
#define VKZG_DEV static inline
#include <cstdio>
#include <cstring>

#include "../../vkzg_amd/csrc/field_fp.h"

using namespace vkzg_amd;

static bool read(Fp &a) {
    for (int i = 0; i < kFpLimbs; i++)
        if (std::scanf("%d", &a.v[i]) != 1) return false;
    return true;
}

int main() {
    char op[32];
    int k;
    while (std::scanf("%31s %d", op, &k) == 2) {
        Fp a, b, c, d, r = fp_zero();
        if (!read(a) || !read(b) || !read(c) || !read(d)) return 1;
        auto is = [&](const char *s) { return std::strcmp(op, s) == 0; };
        if (is("mul")) r = fp_mul(a, b);
        else if (is("sqr")) r = fp_sqr(a);
        else if (is("mul_fold")) r = fp_mul_fold(a, b, c, k);
        else if (is("sqr_fold2")) r = fp_sqr_fold2(a, c, k, d, -2);
        else if (is("mul_sum")) r = fp_mul_sum(a, b, c, d);
        else if (is("norm")) r = fp_norm(a);
        else if (is("norm_wide")) r = fp_norm_wide(a);
        else if (is("triple")) r = fp_triple(a);
        else if (is("inv")) r = fp_inv(a);
        else if (is("canonical")) r = fp_from_digits(fp_canonical(a));
        else if (is("reference")) r = fp_from_digits(fp_mul_reference(a, b));
        else if (is("words")) {
            uint32_t w[12];
            fp_to_words(w, fp_canonical(a));
            r = fp_from_digits(fp_from_words(w));
        } else return 1;
        for (int i = 0; i < kFpLimbs; i++) std::printf("%d ", r.v[i]);
        std::printf("\n");
    }
    return 0;
}
