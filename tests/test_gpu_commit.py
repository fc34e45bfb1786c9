"""Commitments from the multiples table of the setup's 4096 points: single
monomials (each base and each run of terms, digits at the ends of the windows)
against multiples of the setup's own points, and calls on both sides of the
64-blob launch sequence against one-blob calls."""
import random

import pytest

pytestmark = pytest.mark.gpu

R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
W = pow(7, (R - 1) // 4096, R)


def monomials(terms):
    """The blob of sum c X^k over (k, c)."""
    out = [0] * 4096
    for k, c in terms:
        step, x = pow(W, k, R), c % R
        vals = []
        for _ in range(4096):
            vals.append(x)
            x = x * step % R
        for i in range(4096):
            b = int(format(i, "012b")[::-1], 2)
            out[i] = (out[i] + vals[b]) % R
    return b"".join(v.to_bytes(32, "big") for v in out)


def test_monomials(gpu_seeded_prover, seeded_setup_bytes, oracle_mod):
    point = lambda k: seeded_setup_bytes[48 * k:48 * (k + 1)]
    cases = [(k, 1) for k in (0, 1, 63, 64, 65, 127, 2047, 2048, 4031, 4095)]
    # digits -(2^9 - 1), 2^9 and their neighbours in every 10-bit window, the sign, the largest magnitudes
    cases += [(k, c) for k, c in ((5, R - 1), (64, (R - 1) // 2), (700, (R + 1) // 2), (4095, R - 2),
                                  (66, sum(512 << (10 * w) for w in range(20))),
                                  (2, sum(513 << (10 * w) for w in range(20))),
                                  (3, sum(511 << (10 * w) for w in range(20))), (1000, 1 << 253))]
    blobs = b"".join(monomials([c]) for c in cases)
    got = gpu_seeded_prover.blob_to_kzg_commitments(blobs, len(cases))
    for n, (k, c) in enumerate(cases):
        assert got[48 * n:48 * (n + 1)] == oracle_mod.g1_mul(point(k), c % R), (k, hex(c))


@pytest.mark.parametrize("n", [2, 31, 64, 65])
def test_batch_sizes(gpu_seeded_prover, n):
    rng = random.Random(n)
    one = [b"".join(rng.randrange(R).to_bytes(32, "big") for _ in range(4096)) for _ in range(3)]
    pick = [one[(i * i + i // 3) % 3] for i in range(n)]
    single = {b: gpu_seeded_prover.blob_to_kzg_commitments(b, 1) for b in one}
    got = gpu_seeded_prover.blob_to_kzg_commitments(b"".join(pick), n)
    assert got == b"".join(single[b] for b in pick)
