"""Host-buffer copies at the sizes where their shape changes (whole by a kernel
below 3 MiB, in slices by the copy threads from there, of 4 MiB at most; a cell
blob is 256 KiB, a blob 128 KiB), and from input objects that are not bytes:
every blob of a call against its one-blob call, and threads on one prover."""
import random
import threading

import pytest

pytestmark = pytest.mark.gpu

R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
CELLS = 128 * 2048


@pytest.fixture(scope="module")
def ones(gpu_prover):
    rng = random.Random(77)
    out = []
    for _ in range(3):
        blob = b"".join(rng.randrange(R).to_bytes(32, "big") for _ in range(4096))
        cells, proofs = gpu_prover.compute_cells_and_kzg_proofs_batch(blob, 1)
        out.append((blob, cells, proofs))
    return out


@pytest.mark.parametrize("n", [2, 3, 4, 5, 8, 9, 33])
def test_sizes(gpu_prover, ones, n):
    pick = [ones[(i * i + 1) % 3] for i in range(n)]
    blobs, cells, proofs = (b"".join(p[k] for p in pick) for k in range(3))
    assert gpu_prover.compute_cell_kzg_proofs_batch(bytearray(blobs), n) == proofs
    assert gpu_prover.compute_cells_and_kzg_proofs_batch(memoryview(blobs), n) == (cells, proofs)
    present = bytes(1 if (k * 7 + b) % 128 < 64 + b % 5 else 0 for b in range(n) for k in range(128))
    held = bytearray(cells)
    for i, p in enumerate(present):
        if not p:
            held[2048 * i:2048 * (i + 1)] = b"\xaa" * 2048
    assert gpu_prover.recover_cells_batch(held, bytearray(present), n) == cells
    assert gpu_prover.recover_cells_and_kzg_proofs_batch(bytes(held), present, n) == (cells, proofs)


def test_two_threads(gpu_prover, ones):
    bad = []

    def work(k):
        for n in (6, 17, 5):
            pick = [ones[(i + k) % 3] for i in range(n)]
            blobs, cells, proofs = (b"".join(p[j] for p in pick) for j in range(3))
            if gpu_prover.compute_cells_and_kzg_proofs_batch(blobs, n) != (cells, proofs):
                bad.append((k, n))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


# 3 MiB of cells are 12 blobs, of blobs 24; a slice of a third of the copy is 4 MiB
# at 48 and 96 blobs
@pytest.mark.parametrize("n", [11, 12, 13, 23, 24, 25, 32, 47, 48, 49, 97])
def test_sizes_around_the_slices(gpu_prover, ones, n):
    test_sizes(gpu_prover, ones, n)


@pytest.mark.parametrize("n", [11, 12, 24, 25])
def test_threads_on_both_sides_of_a_size(gpu_prover, ones, n):
    """Three threads at once, one with copies of the other shape, every call checked."""
    bad = []

    def work(k):
        for m in (n, 3, n + k, 25):
            pick = [ones[(i + k) % 3] for i in range(m)]
            blobs, cells, proofs = (b"".join(p[j] for p in pick) for j in range(3))
            present = bytes(1 if (c + b) % 2 else 0 for b in range(m) for c in range(128))
            if gpu_prover.compute_cells_and_kzg_proofs_batch(blobs, m) != (cells, proofs):
                bad.append((k, m))
            if gpu_prover.recover_cells_batch(cells, present, m) != cells:
                bad.append((k, m))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
