"""CPU tests of the Python binding's inputs: whatever object they come in, the
library is handed len(object) bytes, and an object whose elements are wider
than a byte is refused, as ctypes buffers of that length refuse it."""
import array
import ctypes

import pytest

import vkzg_amd

BLOB, CELLS = 131072, 262144


class Short:
    """Fewer bytes than its length."""

    def __init__(self, n):
        self.n = n

    def __len__(self):
        return self.n

    def __bytes__(self):
        return b"\x01" * 10


@pytest.fixture
def calls(monkeypatch):
    """A prover on a library that only notes the bytes it is given: (the call's
    inputs by the binding's argument order, the sizes its C side reads)."""
    seen = []

    class Library:
        def __getattr__(self, name):
            sizes, first = {"vkzg_compute_proofs_batch": ((BLOB,), 2), "vkzg_recover_cells_batch": ((CELLS, 128), 2),
                            "vkzg_amd_compute_cells_and_proofs": ((BLOB,), 3),
                            "vkzg_amd_recover_cells_and_proofs": ((CELLS, 128), 3),
                            "vkzg_amd_blob_to_commitments": ((BLOB,), 2),
                            "vkzg_amd_recover_cells_device": ((128,), 4)}[name]

            def call(*args):
                n = args[first + len(sizes)]
                for k, size in enumerate(sizes):
                    ptr = ctypes.cast(args[first + k], ctypes.c_void_p).value
                    assert len(args[first + k]) >= n * size
                    seen.append(ctypes.string_at(ptr, n * size))
                return vkzg_amd.OK

            return call

    monkeypatch.setattr(vkzg_amd, "load", lambda: Library())
    p = object.__new__(vkzg_amd.Prover)
    p._h = None
    mask = bytes([1] * 128)
    yield seen, [(BLOB, lambda x: p.compute_cell_kzg_proofs_batch(x, 1)),
                 (BLOB, lambda x: p.compute_cells_and_kzg_proofs_batch(x, 1)),
                 (BLOB, lambda x: p.blob_to_kzg_commitments(x, 1)),
                 (CELLS, lambda x: p.recover_cells_batch(x, mask, 1)),
                 (CELLS, lambda x: p.recover_cells_and_kzg_proofs_batch(x, mask, 1)),
                 (128, lambda x: p.recover_cells_batch(bytes(CELLS), x, 1)),
                 (128, lambda x: p.recover_cells_and_kzg_proofs_batch(bytes(CELLS), x, 1)),
                 (128, lambda x: p.recover_cells_device(16, 32, 48, x, 1))]


def test_every_entry_point_takes_len_bytes(calls):
    seen, entries = calls
    for n, call in entries:
        data = bytes(i % 251 for i in range(n))
        for x in (data, bytearray(data), memoryview(data), array.array("B", data), list(data)):
            seen.clear()
            call(x)
            assert data in seen, n
        seen.clear()
        call(Short(n))  # never read past its end
        assert b"\x01" * 10 + bytes(n - 10) in seen, n


def test_wider_elements_are_refused(calls):
    seen, entries = calls
    for n, call in entries:
        for x in (array.array("H", [1] * n), memoryview(array.array("I", [1] * n)), array.array("d", [1.0] * n)):
            with pytest.raises(ValueError):
                call(x)
        assert seen == [] or n == 128
        seen.clear()
