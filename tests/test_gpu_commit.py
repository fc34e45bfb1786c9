"""Commitments from the multiples table of the setup's 4096 points: single
monomials (each base and each run of terms, digits at the ends of the windows)
against multiples of the setup's own points, and calls on both sides of the
64-blob launch sequence against one-blob calls."""
import random

import pytest

import vkzg_amd

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


@pytest.mark.parametrize("windows", [28, 31, 36, 42, 51, 63, 85, 127, 0])
def test_smaller_plans(seeded_setup_bytes, oracle_mod, monkeypatch, windows):
    """The tables of a prover with less free memory, and the bucket method of one
    with none to spare (0): digits at the ends of the plan's windows, several
    blobs a call, and calls on both sides of the 64-blob launch sequence."""
    monkeypatch.setenv("VKZG_AMD_COMMIT_WINDOWS", str(windows))
    monkeypatch.setenv("VKZG_AMD_WINDOW", "6")
    n = windows or 24
    c, k = divmod(255, n)
    bits = [w * c + max(0, w - (n - k)) for w in range(n)]
    bits = [b for b in bits if b + c < 250]
    half = 1 << (c - 1)
    point = lambda k: seeded_setup_bytes[48 * k:48 * (k + 1)]
    cases = [(0, 1), (64, R - 1), (4095, (R - 1) // 2), (63, (R + 1) // 2), (1000, 1 << 253)]
    cases += [(65 + i, sum((half + i) << b for b in bits) % R) for i in (-1, 0, 1)]
    with vkzg_amd.Prover(max_batch_size=1, setup_g1_monomial=seeded_setup_bytes) as p:
        one = [monomials([x]) for x in cases]
        got = p.blob_to_kzg_commitments(b"".join(one), len(one))
        want = [oracle_mod.g1_mul(point(k), c % R) for k, c in cases]
        assert [got[48 * n:48 * (n + 1)] for n in range(len(cases))] == want
        assert p.blob_to_kzg_commitments(bytes(131072), 1) == bytes([0xC0]) + bytes(47)
        pick = [(i * i + i // 3) % len(one) for i in range(67)]
        got = p.blob_to_kzg_commitments(b"".join(one[i] for i in pick), 67)
        assert got == b"".join(want[i] for i in pick)
        bad = bytearray(one[0])
        bad[:32] = b"\xff" * 32
        with pytest.raises(vkzg_amd.VkzgError) as e:
            p.blob_to_kzg_commitments(one[1] + bytes(bad), 2)
        assert e.value.code == vkzg_amd.ERR_INVALID_BLOB


@pytest.mark.parametrize("windows", [25, 85])
def test_points_of_order_three(monkeypatch, windows):
    """A setup whose points are all (0, 2), of order 3 on the curve: every run of
    multiples in the tables meets a cancellation and is made again with checked
    additions."""
    monkeypatch.setenv("VKZG_AMD_COMMIT_WINDOWS", str(windows))
    monkeypatch.setenv("VKZG_AMD_WINDOW", "6")
    point = {0: bytes([0xC0]) + bytes(47), 1: bytes([0x80]) + bytes(47), 2: bytes([0xA0]) + bytes(47)}
    cases = [(0, 1), (65, 2), (4095, 3), (7, 511), (8, 512), (9, 513), (10, 1 << 200), (11, 3 << 100), (12, (1 << 253) + 1)]
    with vkzg_amd.Prover(max_batch_size=1, setup_g1_monomial=point[1] * 4096) as p:
        got = p.blob_to_kzg_commitments(b"".join(monomials([x]) for x in cases), len(cases))
    assert [got[48 * n:48 * (n + 1)] for n in range(len(cases))] == [point[c % 3] for _, c in cases]
