"""The doubling chains on quads in homogeneous coordinates (proj_quad.h): the
ladder of batches whose four-lane chains fit the chip and its two conversions,
and the subgroup check on points of every kind of order."""
import random

import pytest

from tests.conftest import random_blob
from tests.test_gpu_verify import _blob_data, _select, g2_setup, verifier  # noqa: F401

pytestmark = pytest.mark.gpu

P = 0x1A0111EA397FE69A4B1BA7B6434BACD764774B84F38512BF6730D2A0F6B0F6241EABFFFEB153FFFFB9FEFFFFFFFFAAAB
R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
G1_INF = b"\xc0" + bytes(47)
GEN_X = 0x17F1D3A73197D7942695638C4FA9AC0FC3688C4F9774B905A14E3A3F171BAC586C55E83FF97A1AEFFB3AF00ADB22C6BB
OMEGA = pow(7, (R - 1) // 4096, R)


def add(p, q):
    if p is None or q is None:
        return p or q
    if p[0] == q[0]:
        if (p[1] + q[1]) % P == 0:
            return None
        lam = 3 * p[0] ** 2 * pow(2 * p[1], -1, P) % P
    else:
        lam = (q[1] - p[1]) * pow(q[0] - p[0], -1, P) % P
    x = (lam * lam - p[0] - q[0]) % P
    return x, (lam * (p[0] - x) - p[1]) % P


def mul(p, k):
    acc = None
    while k:
        if k & 1:
            acc = add(acc, p)
        p, k = add(p, p), k >> 1
    return acc


def sqrt(a):
    y = pow(a, (P + 1) // 4, P)
    return y if y * y % P == a % P else None


def curve_point(rng):
    while True:
        x = rng.randrange(P)
        y = sqrt(x ** 3 + 4)
        if y is not None:
            return x, y


def compress(p):
    b = bytearray(p[0].to_bytes(48, "big"))
    b[0] |= 0x80 | (0x20 if p[1] > (P - 1) // 2 else 0)
    return bytes(b)


def monomial(e):
    """X^e in the blob's order (bit-reversed roots of unity)."""
    brev = [int(format(i, "012b")[::-1], 2) for i in range(4096)]
    return b"".join(pow(OMEGA, e * k % 4096, R).to_bytes(32, "big") for k in brev)


# quads into XYZZ points (up to 8 blobs), quads normalised, pairs normalised
@pytest.mark.parametrize("n", [1, 5, 8, 9, 67, 128, 129])
def test_ladder_degenerate_blobs(gpu_prover, rng, n):
    # the quotients of 0 and 5 by X^64 - h are 0, that of X^64 is 1
    kinds = [(bytes(131072), G1_INF), ((5).to_bytes(32, "big") * 4096, G1_INF),
             (monomial(64), compress((GEN_X, min(sqrt(GEN_X ** 3 + 4), P - sqrt(GEN_X ** 3 + 4))))),
             (random_blob(rng), None)]
    pick = [kinds[(n + i) % 4] for i in range(n)]
    got = gpu_prover.compute_cell_kzg_proofs_batch(b"".join(b for b, _ in pick), n)
    rand = gpu_prover.compute_cell_kzg_proofs_batch(kinds[3][0], 1)
    for i, (_, want) in enumerate(pick):
        assert got[6144 * i:6144 * (i + 1)] == (want * 128 if want is not None else rand), i


def _bad_points():
    rng = random.Random(5)
    q = curve_point(rng)
    three = (0, 2)                         # order 3
    cof = mul(q, R)                        # order divides the cofactor
    h = 0x396C8C005555E1568C00AAAB0000AAAB
    good = mul(q, h)                       # in the group
    assert mul(good, R) is None and mul(three, 3) is None
    return {"random": q, "order3": three, "order3_neg": (0, P - 2), "cofactor": cof,
            "good_plus_order3": add(good, three), "good_plus_cofactor": add(good, cof),
            "cofactor_plus_order3": add(cof, three)}, good


@pytest.mark.parametrize("n", [2, 17])
def test_subgroup_check(verifier, rng, n):  # noqa: F811
    import vkzg_amd
    bad, good = _bad_points()
    cells, proofs, coms = _blob_data(verifier, random_blob(rng), 1)
    c, idx, ce, pr = _select(cells, proofs, coms, [(0, k) for k in range(n)])
    pr = bytes(pr)
    assert verifier.verify_cell_kzg_proof_batch(c, idx, ce, pr)
    # a point of the group that is no proof of this cell: checked, and false
    assert not verifier.verify_cell_kzg_proof_batch(c, idx, ce, pr[:-48] + compress(good))
    for name, q in bad.items():
        for at in (0, n - 1):
            with pytest.raises(vkzg_amd.VkzgError) as e:
                verifier.verify_cell_kzg_proof_batch(c, idx, ce, pr[:48 * at] + compress(q) + pr[48 * at + 48:])
            assert e.value.code == vkzg_amd.ERR_BADARGS, name
