"""The two-step blob transform in front of phase A (fk20_scalars.hip): elements at
the edges of its waves' columns, on both launch shapes (two waves per four
columns up to 32 blobs on 256 CUs, one above), for whole proofs and for the
canonical check."""
import pytest

from tests.conftest import SEEDED_TAU

pytestmark = pytest.mark.gpu

R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
SPOTS = [0, 3, 4, 63, 64, 255, 256, 2047, 2048, 4031, 4095]


def _single(i, value):
    return bytes(32 * i) + value.to_bytes(32, "big") + bytes(32 * (4095 - i))


@pytest.mark.parametrize("n", [1, 33])
def test_noncanonical_element_anywhere(gpu_prover, n):
    import vkzg_amd
    zero = bytes(131072)
    for k, i in enumerate(SPOTS):
        at = k * 7 % n
        for value, ok in ((R - 1, True), (R, False), (2 ** 256 - 1, False)):
            blobs = zero * at + _single(i, value) + zero * (n - 1 - at)
            if ok:
                gpu_prover.compute_cell_kzg_proofs_batch(blobs, n)
                continue
            with pytest.raises(vkzg_amd.VkzgError) as e:
                gpu_prover.compute_cell_kzg_proofs_batch(blobs, n)
            assert e.value.code == vkzg_amd.ERR_INVALID_BLOB


@pytest.mark.parametrize("n", [len(SPOTS), 44])
def test_single_elements_against_closed_form(gpu_seeded_prover, oracle_mod, n):
    # one nonzero value per blob: its proofs depend on every output of the transform
    blobs = [_single(i, R - 1 - i) for i in SPOTS]
    want = []
    for b in blobs:
        rc, proofs = oracle_mod.proofs_from_tau(b, SEEDED_TAU)
        assert rc == 0
        want.append(proofs)
    got = gpu_seeded_prover.compute_cell_kzg_proofs_batch(b"".join(blobs[k % len(SPOTS)] for k in range(n)), n)
    for k in range(n):
        assert got[6144 * k:6144 * (k + 1)] == want[k % len(SPOTS)], k
