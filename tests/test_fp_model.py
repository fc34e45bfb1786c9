"""CPU test of the device's Fp form (vkzg_amd/csrc/field_fp.h, 13 signed limbs
of 30 bits), compiled for the host with g++ -ftrapv: every operation against
Python integers on random values and on operands whose limbs sit at the ends
of their classes (N: 2^29 + 8 in magnitude, N2: twice that), where a column
comes nearest to overflowing."""
import os
import random
import subprocess

import pytest

P = 0x1A0111EA397FE69A4B1BA7B6434BACD764774B84F38512BF6730D2A0F6B0F6241EABFFFEB153FFFFB9FEFFFFFFFFAAAB
RINV = pow(1 << 390, -1, P)
HERE = os.path.dirname(os.path.abspath(__file__))
N, N2, TOP = (1 << 29) + 8, (1 << 30) + 16, 1 << 24


def value(l):
    return sum(v << (30 * i) for i, v in enumerate(l))


def balanced(x):
    out = []
    for _ in range(12):
        v = x & ((1 << 30) - 1)
        v -= (v >> 29) << 30
        out.append(v)
        x = (x - v) >> 30
    return out + [x]


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("fp") / "fp_host")
    subprocess.run(["g++", "-O1", "-ftrapv", "-std=c++17", "-o", exe, os.path.join(HERE, "c", "fp_host.cpp")], check=True)

    def run(cases):
        text = "\n".join(" ".join([op, str(k)] + [str(v) for o in ops for v in o]) for op, k, ops in cases)
        out = subprocess.run([exe], input=text + "\n", capture_output=True, text=True, check=True).stdout
        rows = [[int(v) for v in line.split()] for line in out.splitlines()]
        assert len(rows) == len(cases)
        return rows

    return run


def operands(rng, bound):
    """Random residues, and limbs at the ends of their class with every sign pattern that lines columns up."""
    out = [balanced(rng.randrange(-8 * P, 8 * P)) for _ in range(40)] if bound == N else [
        [x + y for x, y in zip(balanced(rng.randrange(-4 * P, 4 * P)), balanced(rng.randrange(-4 * P, 4 * P)))]
        for _ in range(40)]
    for pattern in ([1] * 13, [-1] * 13, [(-1) ** i for i in range(13)], [rng.choice((-1, 1)) for _ in range(13)]):
        out.append([s * bound for s in pattern[:12]] + [pattern[12] * TOP])
    return out + [[0] * 13, balanced(1), balanced(P - 1), balanced(-P)]


def strict(r):
    return all(-(1 << 29) <= v < 1 << 29 for v in r[:12])


def test_products(host):
    rng = random.Random(30)
    z = [0] * 13
    cases = []
    for a in operands(rng, N2):
        for b in operands(rng, N):
            cases.append(("mul", 0, (a, b, z, z)))
    wide = [[s * ((1 << 31) - 1) for s in (1, -1) * 6] + [TOP], balanced(5 * P)]
    for a in operands(rng, N):
        cases.append(("sqr", 0, (a, z, z, z)))
        for c in wide:
            cases.append(("mul_fold", rng.choice((-8, -4, -1, 1)), (a, rng.choice(operands(rng, N)), c, z)))
            cases.append(("sqr_fold2", -1, (a, z, c, rng.choice(operands(rng, N)))))
        for _ in range(8):
            o = operands(rng, N)
            cases.append(("mul_sum", 0, (a, rng.choice(o), rng.choice(o), rng.choice(o))))
    # every column at the end of its class at once
    e = [N] * 12 + [TOP]
    cases.append(("mul_sum", 0, (e, e, e, e)))
    cases.append(("mul_sum", 0, (e, [-v for v in e], e, [-v for v in e])))
    for (op, k, (a, b, c, d)), r in zip(cases, host(cases)):
        a, b, c, d = value(a), value(b), value(c), value(d)
        add = 0
        if op == "mul":
            prod = a * b
        elif op == "sqr":
            prod = a * a
        elif op == "mul_fold":
            prod, add = a * b, k * c
        elif op == "sqr_fold2":
            prod, add = a * a, k * c - 2 * d
        else:
            prod = a * b + c * d
        assert strict(r), (op, r)
        v = value(r) - add
        assert (v - prod * RINV) % P == 0, op
        # the stated magnitude: |product| / R + p / 2, and a little for the rounding digits
        assert abs(v) <= abs(prod) // (1 << 390) + P // 2 + (P >> 27), op
        if prod % P == 0 and abs(prod) <= 256 * P * P:
            assert v == 0, op


def test_carry_passes(host):
    rng = random.Random(31)
    z = [0] * 13
    cases = []
    for _ in range(200):
        lim = 3 * (1 << 29) - 1
        cases.append(("norm", 0, ([rng.choice((-lim, lim, rng.randint(-lim, lim))) for _ in range(12)] + [rng.randint(-TOP, TOP)], z, z, z)))
        cases.append(("norm_wide", 0, ([rng.choice((-(1 << 31), (1 << 31) - 1, rng.randint(-(1 << 31), (1 << 31) - 1)))
                                        for _ in range(12)] + [rng.randint(-TOP, TOP)], z, z, z)))
        ends = (-(1 << 29), (1 << 29) - 1)
        cases.append(("triple", 0, ([rng.choice(ends + (rng.randint(*ends),)) for _ in range(12)] + [rng.randint(-TOP, TOP)], z, z, z)))
    for (op, _, (a, _, _, _)), r in zip(cases, host(cases)):
        assert value(r) == value(a) * (3 if op == "triple" else 1), op
        assert all(abs(v) <= N for v in r[:12]), op


def test_canonical_inverse_words_and_reference(host):
    rng = random.Random(32)
    z = [0] * 13
    vals = [0, 1, -1, P - 1, 1 - P, P // 2, -(P // 2)] + [rng.randrange(-P + 1, P) for _ in range(300)]
    rows = host([("canonical", 0, (balanced(v), z, z, z)) for v in vals])
    assert [value(r) for r in rows] == [v % P for v in vals]
    assert all(0 <= d < 1 << 30 for r in rows for d in r)
    rows = host([("words", 0, (balanced(v), z, z, z)) for v in vals])
    assert [value(r) for r in rows] == [v % P for v in vals]
    R = 1 << 390
    inv = vals + [P, -P, 2 * P, 7 * P + 3, -9 * P - 1]
    for v, r in zip(inv, host([("inv", 0, (balanced(v), z, z, z)) for v in inv])):
        # (x R)^-1 -> x^-1 R
        assert value(r) % P == (pow(v, -1, P) * R * R % P if v % P else 0)
    pairs = [(rng.randrange(-4 * P, 4 * P), rng.randrange(-4 * P, 4 * P)) for _ in range(100)]
    for (x, y), r in zip(pairs, host([("reference", 0, (balanced(x), balanced(y), z, z)) for x, y in pairs])):
        assert value(r) == x * y * RINV % P
