"""CPU test of the sum an Fp12 product ends in (vkzg_amd/csrc/fp12_tree.h),
compiled for the host with g++ -ftrapv and run on 32 threads as lanes: terms
whose limbs sit at the ends of what two products add up to ([-2^30, 2^30)), and
at the places where a carry pass leaves the largest limbs."""
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
TOP = 1 << 24


def value(l):
    return sum(v << (30 * i) for i, v in enumerate(l))


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("fp12") / "fp12_tree_host")
    subprocess.run(["g++", "-O1", "-ftrapv", "-std=c++17", "-pthread", "-o", exe,
                    os.path.join(HERE, "c", "fp12_tree_host.cpp")], check=True)

    def run(cases):
        text = "\n".join(" ".join(str(v) for term in c for part in term for v in part) for c in cases)
        r = subprocess.run([exe], input=text + "\n", capture_output=True, text=True)
        assert r.returncode == 0, (r.returncode, r.stdout.count("\n"))
        return [[int(v) for v in line.split()] for line in r.stdout.splitlines()]

    return run


def test_limbs_at_the_ends(host):
    rng = random.Random(12)
    lo, hi = -(1 << 30), (1 << 30) - 1
    # halves of the sums of two terms whose carry pass leaves a digit at an end of
    # its range and hands the largest carries on
    ends = [lo, hi, hi - 1, 3 << 28, (3 << 28) - 1, -(3 << 28), -(3 << 28) - 1, 1 << 28, (1 << 28) - 1, -(1 << 28), 0]
    cases = []
    for a in ends:
        for b in ends:  # every term the same, limbs alternating
            part = [a if i % 2 else b for i in range(12)] + [TOP]
            cases.append([[part, [-v - 1 for v in part[:12]] + [-TOP]]] * 6)
    # digits at the end of their range with the largest carries below them, for every
    # way two pairs of terms and two single ones may meet in a pass
    for sign in (1, -1):
        for s in range(6):
            for t in range(s):
                rest = [k for k in range(6) if k not in (s, t)]
                for mate in rest[1:]:
                    pairs = {rest[0]: 0, mate: 1}
                    pairs.update(zip([k for k in rest if k not in pairs], (0, 1)))
                    low = (hi, 1 << 29) if sign > 0 else (lo, -(1 << 29) - 1)
                    top = {0: 1 << 28, 1: (1 << 28) - 1, None: (1 << 29) - 1} if sign > 0 else \
                        {0: -(1 << 28), 1: -(1 << 28), None: -(1 << 29)}
                    cases.append([[[low[k not in pairs], top[pairs.get(k)]] * 6 + [sign * TOP]] * 2 for k in range(6)])
    for _ in range(150):
        cases.append([[[rng.choice(ends + [rng.randint(lo, hi)]) for _ in range(12)] + [rng.randint(-TOP, TOP)]
                       for _ in range(2)] for _ in range(6)])
    rows = host(cases)
    assert len(rows) == len(cases)
    for c, r in zip(cases, rows):
        for k in range(2):
            got = r[13 * k:13 * k + 13]
            assert value(got) == sum(value(t[k]) for t in c)
            assert all(abs(v) <= (1 << 29) + 8 for v in got[:12])  # an operand of the next product
