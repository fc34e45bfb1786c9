#!/usr/bin/env python3
"""Writes constants.h: BLS12-381 Fp/Fr Montgomery constants as 32-bit limbs.

Every value is derived here from p, r and the coset shift 7 with Python big
integers, so the header is reproducible:  python3 gen_constants.py > constants.h
"""

P = 0x1A0111EA397FE69A4B1BA7B6434BACD764774B84F38512BF6730D2A0F6B0F6241EABFFFEB153FFFFB9FEFFFFFFFFAAAB
R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
FP_LIMBS, FP_BITS = 13, 30  # Fp in registers: 13 signed limbs of 30 bits
RP = 1 << (FP_LIMBS * FP_BITS)  # Montgomery radix for Fp, 2^390
GCD_LIMBS, GCD_BITS = 14, 28  # Fp inside the binary-GCD inversion
RR = 1 << 256  # Montgomery radix for Fr
# Endomorphism constants of BLS12-381 G1: beta is a cube root of unity in Fp,
# lambda the matching cube root of unity in Fr with phi(x, y) = (beta*x, y) = lambda*P.
BETA = 0x1A0111EA397FE699EC02408663D4DE85AA0D857D89759AD4897D29650FB85F9B409427EB4F49FFFD8BFD00000000AAAC


Z_ABS = 0xD201000000010000  # |z|, z = -0xd201000000010000 is the BLS parameter
LAMBDA = Z_ABS * Z_ABS - 1  # z^2 - 1: phi(P) = [LAMBDA]P on G1, r = LAMBDA^2 + LAMBDA + 1


# The model 3 Y^2 Z = 2 X^3 - Z^3 of proj_quad.h: SIGMA^2 = -12, NU^3 = 3 SIGMA / 2
SIGMA = pow(-12, (P + 1) // 4, P)


def cbrt(a):
    """A cube root of a cube mod P, from the 3-part of P - 1 and a non-cube."""
    s, t = 0, P - 1
    while t % 3 == 0:
        s, t = s + 1, t // 3
    g = next(g for g in range(2, 100) if pow(g, (P - 1) // 3, P) != 1)
    c = pow(g, t, P)  # of order 3^s
    x = pow(a, pow(3, -1, t), P)  # x^3 = a e with e of order dividing 3^(s-1)
    for k in range(3 ** (s - 1)):
        y = x * pow(c, k, P) % P
        if pow(y, 3, P) == a % P:
            return y
    raise ValueError("not a cube")


NU = cbrt(3 * SIGMA * pow(2, -1, P))


def f2mul(a, b):
    return ((a[0] * b[0] - a[1] * b[1]) % P, (a[0] * b[1] + a[1] * b[0]) % P)


def f2pow(a, e):
    r = (1, 0)
    while e:
        if e & 1:
            r = f2mul(r, a)
        a = f2mul(a, a)
        e >>= 1
    return r


def limbs(x, n):
    return [(x >> (32 * i)) & 0xFFFFFFFF for i in range(n)]


def arr(name, x, n):
    body = ", ".join("0x%08xu" % v for v in limbs(x, n))
    return "constexpr uint32_t %s[%d] = {%s};" % (name, n, body)


def arr30(name, x):
    """x in balanced limbs: 30-bit digits in [-2^29, 2^29), the top one what remains."""
    assert 0 <= x < 1 << (FP_LIMBS * FP_BITS - 2)
    d = []
    for _ in range(FP_LIMBS - 1):
        v = x & ((1 << FP_BITS) - 1)
        if v >> (FP_BITS - 1):
            v -= 1 << FP_BITS
        d.append(v)
        x = (x - v) >> FP_BITS
    d.append(x)
    return "constexpr int32_t %s[%d] = {%s};" % (name, FP_LIMBS, ", ".join("%d" % v for v in d))


def arr_digits(name, x, n, bits):
    """x in n unsigned digits of that many bits."""
    assert 0 <= x < 1 << (n * bits)
    body = ", ".join("0x%xu" % ((x >> (bits * i)) & ((1 << bits) - 1)) for i in range(n))
    return "constexpr uint32_t %s[%d] = {%s};" % (name, n, body)


def main():
    out = []
    out.append("// Generated by gen_constants.py -- BLS12-381 field constants, little-endian limbs:")
    out.append("// Fp values in balanced 30-bit limbs (13 of them, Montgomery radix 2^390), Fp")
    out.append("// exponents and all Fr values in 32-bit limbs.")
    out.append("#pragma once")
    out.append("#include <cstdint>")
    out.append("namespace vkzg_amd {")
    out.append("namespace cfp {")
    out.append(arr30("P", P))
    out.append("constexpr uint32_t N0 = 0x%xu;  // -p^-1 mod 2^32" % ((-pow(P, -1, 1 << 32)) % (1 << 32)))
    out.append(arr30("ONE", RP % P))
    out.append(arr30("R2", RP * RP % P))
    out.append(arr30("FOUR_M", 4 * RP % P))
    out.append(arr30("BETA_M", BETA * RP % P))
    assert SIGMA * SIGMA % P == P - 12 and 2 * pow(NU, 3, P) % P == 3 * SIGMA % P
    out.append(arr30("SIGMA_M", SIGMA * RP % P))
    out.append(arr30("INV_SIGMA_M", pow(SIGMA, -1, P) * RP % P))
    out.append(arr30("NU_M", NU * RP % P))
    out.append(arr30("SIGMA_OVER_NU_M", SIGMA * pow(NU, -1, P) * RP % P))
    out.append(arr30("NU_BETA_M", NU * BETA * RP % P))
    out.append(arr30("NU_BETA2_M", NU * BETA * BETA * RP % P))
    out.append(arr30("R3_M", RP ** 3 % P))  # Montgomery form of R^2: turns a plain inverse of xR into x^-1 R
    # 2^384 mod p as a plain value: a Montgomery product of x R by it gives
    # x 2^384 mod p, the reference's 12 x 32-bit Montgomery form (tables file v1)
    out.append(arr30("REF_R", (1 << 384) % P))
    out.append("// p and (p - 1) / 2 in unsigned 30-bit digits")
    out.append(arr_digits("PU", P, FP_LIMBS, FP_BITS))
    out.append(arr_digits("HALFU", (P - 1) // 2, FP_LIMBS, FP_BITS))
    out.append("// p, -p^-1 mod 2^28 and 32p in the 28-bit limbs of the binary-GCD inversion")
    out.append(arr_digits("GCD_P", P, GCD_LIMBS, GCD_BITS))
    out.append("constexpr uint32_t GCD_N0 = 0x%07xu;" % ((-pow(P, -1, 1 << GCD_BITS)) % (1 << GCD_BITS)))
    out.append(arr_digits("GCD_P32", 32 * P, GCD_LIMBS, GCD_BITS))  # makes the signed GCD result non-negative
    out.append("// exponents, 32-bit words")
    out.append(arr("P_MINUS_2", P - 2, 12))
    out.append(arr("SQRT_EXP", (P + 1) // 4, 12))
    out.append(arr("P_MINUS_3_DIV_4", (P - 3) // 4, 12))
    out.append(arr("P_MINUS_1_DIV_2", (P - 1) // 2, 12))
    # Frobenius of Fp12 = Fp2[w]/(w^6 - xi): (a w^m)^p = conj(a) FROB1_m w^m and
    # (a w^m)^(p^2) = a FROB2_m w^m with FROB1_m = xi^(m(p-1)/6) in Fp2 and
    # FROB2_m = xi^(m(p^2-1)/6), which lies in Fp.
    assert (P - 1) % 6 == 0
    for m in range(6):
        g1 = f2pow((1, 1), m * (P - 1) // 6)
        g2 = f2pow((1, 1), m * (P * P - 1) // 6)
        assert g2[1] == 0
        out.append(arr30("FROB1_%d_C0" % m, g1[0] * RP % P))
        out.append(arr30("FROB1_%d_C1" % m, g1[1] * RP % P))
        out.append(arr30("FROB2_%d" % m, g2[0] * RP % P))
    out.append("}  // namespace cfp")
    out.append("namespace cfr {")
    out.append(arr("P", R, 8))
    out.append("constexpr uint32_t N0 = 0x%08xu;" % ((-pow(R, -1, 1 << 32)) % (1 << 32)))
    out.append(arr("ONE", RR % R, 8))
    out.append(arr("R2", RR * RR % R, 8))
    out.append(arr("P_MINUS_2", R - 2, 8))
    w = pow(7, (R - 1) // 8192, R)
    out.append(arr("OMEGA8192_M", w * RR % R, 8))
    out.append(arr("OMEGA8192_INV_M", pow(w, -1, R) * RR % R, 8))
    out.append(arr("SEVEN_M", 7 * RR % R, 8))
    out.append(arr("INV_SEVEN_M", pow(7, -1, R) * RR % R, 8))
    out.append(arr("INV_4096_M", pow(4096, -1, R) * RR % R, 8))
    out.append(arr("INV_8192_M", pow(8192, -1, R) * RR % R, 8))
    out.append(arr("SEVEN_POW64_M", pow(7, 64, R) * RR % R, 8))
    # prod over all 128-th roots w of (y - w) = y^128 - 1 = 7^8192 - 1 for every
    # y = 7^64 omega_128^k; its inverse turns 1/z(y) into a product.
    k = (pow(7, 8192, R) - 1) % R
    assert k != 0
    out.append(arr("INV_SEVEN_POW8192_MINUS_1_M", pow(k, -1, R) * RR % R, 8))
    out.append(arr("INV_64_M", pow(64, -1, R) * RR % R, 8))
    # GLV split k = k1 + LAMBDA k2 of a scalar k < r: k2 = floor(k / LAMBDA) by
    # Barrett reduction with GLV_MU = floor(2^256 / LAMBDA) (129 bits)
    assert R == LAMBDA * LAMBDA + LAMBDA + 1 and LAMBDA.bit_length() == 128
    out.append(arr("GLV_LAMBDA", LAMBDA, 4))
    out.append(arr("GLV_MU", (1 << 256) // LAMBDA, 5))
    out.append("}  // namespace cfr")
    out.append("constexpr uint64_t kZAbs = 0x%xull;  // |z| of BLS12-381 (z < 0)" % Z_ABS)
    out.append("}  // namespace vkzg_amd")
    # Self-checks on the endomorphism constant.
    assert pow(BETA, 3, P) == 1 and BETA != 1
    print("\n".join(out))


if __name__ == "__main__":
    main()
