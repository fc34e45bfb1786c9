"""Phase A's shares (runs of terms x window groups, chosen by batch size) and
the sums over them: proofs of batches at the sizes where the shape changes, and
of fixed group counts that divide nothing evenly, bit-exact against the
consensus vectors.  Each MSM's lanes, and a wave's mix of blobs and bases, move
with the batch size, so every blob of the batch is compared."""
import pytest

import vkzg_amd

pytestmark = pytest.mark.gpu


def batch(vectors, n):
    names = vectors.valid_compute()
    pick = [names[(3 * i + i // 7) % len(names)] for i in range(n)]
    return b"".join(vectors.blob(x) for x in pick), b"".join(vectors.proofs(x) for x in pick)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 8, 9, 17, 22, 33, 65, 100, 129, 255])
def test_fitted_shares(gpu_prover, vectors, n):
    blobs, want = batch(vectors, n)
    assert 1 <= gpu_prover.get_tuning(n)["phase_a_groups"] <= 20
    assert gpu_prover.compute_cell_kzg_proofs_batch(blobs, n) == want


@pytest.mark.parametrize("groups,splits,ladder", [(3, 1, 1), (7, 1, 4), (19, 1, 2), (20, 3, 4), (13, 2, 1)])
def test_fixed_groups(gpu_prover, vectors, groups, splits, ladder):
    saved = gpu_prover.get_tuning(11)
    blobs, want = batch(vectors, 11)
    try:
        gpu_prover.set_tuning(11, phase_a_groups=groups, splits=splits, ladder_splits=ladder)
        assert gpu_prover.compute_cell_kzg_proofs_batch(blobs, 11) == want
    finally:
        gpu_prover.set_tuning(11, **saved)


def test_smallest_prover(vectors, monkeypatch):
    """max_batch_size 1: the partials have the room of a few blobs all the same."""
    monkeypatch.setenv("VKZG_AMD_WINDOW", "8")
    with vkzg_amd.Prover(max_batch_size=1) as p:
        blobs, want = batch(vectors, 2)
        assert p.compute_cell_kzg_proofs_batch(blobs, 2) == want


@pytest.mark.parametrize("cap", [1, 3])
def test_slots_without_room_to_spare(gpu_prover, vectors, cap):
    """A server whose budget leaves its slots no room beside their working sets:
    phase A's partials reach into the memory of the buckets."""
    info = gpu_prover.info()
    with vkzg_amd.Server(gpu_prover, batch_blobs=1, slots=1) as one:
        per_blob = one.stats()["slot_bytes"]
    with vkzg_amd.Server(gpu_prover, batch_blobs=cap, slots=1,
                         hbm_budget_bytes=info["resident_table_bytes"] + cap * per_blob) as srv:
        assert srv.stats()["batch_blobs"] == cap
        for n in (1, 2, cap, 7):
            blobs, want = batch(vectors, n)
            for _ in range(3):  # captured, then replayed
                assert srv.wait(srv.submit_proofs(blobs, n))[0] == want
