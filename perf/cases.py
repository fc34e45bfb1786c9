"""The work a node or builder has this library do, as cases that can be timed.

A case is one pass through the public Python entry points on one long-lived
prover (the library's defaults, as a program gets them without tuning).  The
setup is tests/golden/seeded_setup.bin, because it has the G2 side that
verification needs; no time depends on which setup it is.

Kinds:
  proofs          compute_cell_kzg_proofs_batch on host buffers (encode)
  proofs_device   the same on blobs and proofs that stay in GPU memory
  cells_proofs    compute_cells_and_kzg_proofs_batch (extension and proofs)
  recover         recover_cells_batch on host buffers (decode)
  recover_device  the same on cells that stay in GPU memory
  recover_proofs  recover_cells_and_kzg_proofs_batch
  verify          verify_cell_kzg_proof_batch, a few messages one after another
  commit          blob_to_kzg_commitments

`present` says which cells of a blob a recovery holds: "half", exactly 64 at
random, or "ragged", 64 to 127 at random, other ones in each blob.
"""
import math
import os

import numpy as np
import torch  # before the library: both then share torch's HIP runtime

import vkzg_amd

SETUP = os.path.join("tests", "golden", "seeded_setup.bin")
BLOB, CELLS, PROOFS, CELL = 131072, 262144, 6144, 2048
MESSAGES = 4  # verification messages of one pass; a seed's bits say which are tampered with
FP, FR = 300, 136  # 32-bit multiply-adds of one Fp and one Fr product
# Products of one blob: 128 sums of 64 points by 18 windows, the two halves of
# the second transform over G1 and its bucket sums; recovery's transforms.
PROOF_OPS = 2 * FP * 2_960_000
RECOVER_OPS = 2 * FR * 200_000
EXTEND_OPS = 2 * FR * 100_000
VERIFY_CELL_OPS = 2 * FP * 5_000  # decompression, group membership and the sums, of one cell
VERIFY_CALL_OPS = 2 * FP * 100_000  # the pairing check
COMMIT_OPS = 2 * FP * 4096 * 250

_prover = None


def prover():
    """The prover such a program makes once and keeps."""
    global _prover
    if _prover is None:
        data = open(SETUP, "rb").read()
        _prover = vkzg_amd.Prover(setup_g1_monomial=data[: 4096 * 48])
        _prover.load_g2_setup(data[4096 * 48:])
    return _prover


def listed():
    return [
        # one blob for a transaction pool or a proposer: latency of the smallest call
        {"name": "proofs_1", "kind": "proofs", "blobs": 1},
        # one block's blobs (an odd count)
        {"name": "proofs_9", "kind": "proofs", "blobs": 9},
        # a builder's batch through host memory
        {"name": "proofs_64", "kind": "proofs", "blobs": 64},
        # bulk proving with everything resident: the benchmark's workload
        {"name": "proofs_256_device", "kind": "proofs_device", "blobs": 256},
        # a block's data columns made from its blobs
        {"name": "cells_proofs_21", "kind": "cells_proofs", "blobs": 21},
        # one blob rebuilt from half of its cells
        {"name": "recover_1", "kind": "recover", "blobs": 1, "present": "half"},
        # a block's blobs rebuilt through host memory, each missing other cells
        {"name": "recover_37", "kind": "recover", "blobs": 37, "present": "ragged"},
        # the benchmark's recovery: 64 blobs in GPU memory, exactly half present
        {"name": "recover_64_device", "kind": "recover_device", "blobs": 64, "present": "half"},
        # a node that rebuilds a block's columns and serves them with proofs
        {"name": "recover_proofs_6", "kind": "recover_proofs", "blobs": 6, "present": "ragged"},
        # column messages of a block as they arrive: the small verification
        {"name": "verify_128", "kind": "verify", "cells": 128},
        # everything of a large block, or of many blocks while syncing
        {"name": "verify_8192", "kind": "verify", "cells": 8192},
        # commitments of a builder's batch
        {"name": "commit_64", "kind": "commit", "blobs": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["proofs", "proofs", "proofs_device", "cells_proofs", "recover", "recover_device", "recover_proofs",
                       "verify", "commit"])
    if kind == "verify":
        return {"kind": kind, "cells": _log(rng, 1, 8192)}
    top = {"proofs": 192, "proofs_device": 255, "cells_proofs": 128, "recover": 128, "recover_device": 256,
           "recover_proofs": 64, "commit": 64}[kind]
    c = {"kind": kind, "blobs": _log(rng, 1, top)}
    if kind.startswith("recover"):
        c["present"] = rng.choice(["half", "ragged"])
    return c


def _blobs(rng, n):
    """n blobs of 4096 field elements, the whole 32 bytes in use, below the modulus."""
    b = rng.integers(0, 256, size=(n, 4096, 32), dtype=np.uint8)
    b[:, :, 0] %= 0x73
    return b.tobytes()


def _present(rng, n, how):
    m = np.zeros((n, 128), dtype=np.uint8)
    for row in m:
        k = 64 if how == "half" else int(rng.integers(64, 128))
        row[rng.permutation(128)[:k]] = 1
    return m


def _erased(cells, present):
    c = np.frombuffer(cells, dtype=np.uint8).reshape(-1, 128, CELL).copy()
    c[present == 0] = 0
    return c.tobytes()


def _messages(rng, seed, cells):
    """MESSAGES verification messages: the same cells, one field element changed where the seed's bit is set."""
    p = prover()
    n = min(64, -(-cells // 128))
    blobs = _blobs(rng, n)
    ext, proofs = p.compute_cells_and_kzg_proofs_batch(blobs, n)
    coms = np.frombuffer(p.blob_to_kzg_commitments(blobs, n), dtype=np.uint8).reshape(n, 48)
    at = rng.permutation(128 * n)[:cells]
    ext = np.frombuffer(ext, dtype=np.uint8).reshape(-1, CELL)[at]
    proofs = np.frombuffer(proofs, dtype=np.uint8).reshape(-1, 48)[at].tobytes()
    indices = [int(k) % 128 for k in at]
    coms = coms[at // 128].tobytes()
    good = ext.tobytes()
    made = []
    for k in range(MESSAGES):
        mine = good
        if (seed >> k) & 1:
            bad = bytearray(good)
            bad[CELL * int(rng.integers(cells)) + 31] ^= 1
            mine = bytes(bad)
        made.append((coms, indices, mine, proofs))
    return made


def prepare(case, seed):
    rng = np.random.default_rng([seed, 20261202])
    kind, n = case["kind"], case.get("blobs", 0)
    p = prover()
    s = {"kind": kind, "n": n, "prover": p}
    if kind == "verify":
        s["messages"] = _messages(rng, seed, case["cells"])
        return s
    blobs = _blobs(rng, n)
    if not kind.startswith("recover"):
        if kind == "proofs_device":
            s["in"] = torch.frombuffer(bytearray(blobs), dtype=torch.uint8).cuda()
            s["out"] = torch.empty(n * PROOFS, dtype=torch.uint8, device="cuda")
        else:
            s["in"] = blobs
        return s
    present = _present(rng, n, case["present"])
    cells = _erased(p.compute_cells_and_kzg_proofs_batch(blobs, n)[0], present)
    s["present"] = present.tobytes()
    if kind == "recover_device":
        s["in"] = torch.frombuffer(bytearray(cells), dtype=torch.uint8).cuda()
        s["d_present"] = torch.from_numpy(present).cuda()
        s["out"] = torch.empty(n * CELLS, dtype=torch.uint8, device="cuda")
    else:
        s["in"] = cells
    return s


def run(s):
    p, n, kind = s["prover"], s["n"], s["kind"]
    if kind == "proofs":
        return np.frombuffer(p.compute_cell_kzg_proofs_batch(s["in"], n), dtype=np.uint8)
    if kind == "proofs_device":
        p.compute_proofs_device(s["out"].data_ptr(), s["in"].data_ptr(), n)
        return s["out"]
    if kind == "cells_proofs":
        return [np.frombuffer(b, dtype=np.uint8) for b in p.compute_cells_and_kzg_proofs_batch(s["in"], n)]
    if kind == "recover":
        return np.frombuffer(p.recover_cells_batch(s["in"], s["present"], n), dtype=np.uint8)
    if kind == "recover_device":
        p.recover_cells_device(s["out"].data_ptr(), s["in"].data_ptr(), s["d_present"].data_ptr(), s["present"], n)
        return s["out"]
    if kind == "recover_proofs":
        got = p.recover_cells_and_kzg_proofs_batch(s["in"], s["present"], n)
        return [np.frombuffer(b, dtype=np.uint8) for b in got]
    if kind == "verify":
        return [p.verify_cell_kzg_proof_batch(*m) for m in s["messages"]]
    return np.frombuffer(p.blob_to_kzg_commitments(s["in"], n), dtype=np.uint8)


def work(case):
    """Inputs read once and outputs written once; field products as 32-bit multiply-adds, two operations each."""
    kind, n = case["kind"], case.get("blobs", 0)
    if kind == "verify":
        c = case["cells"]
        return {"bytes": MESSAGES * c * (48 + 8 + CELL + 48), "flops": MESSAGES * (c * VERIFY_CELL_OPS + VERIFY_CALL_OPS)}
    if kind in ("proofs", "proofs_device"):
        return {"bytes": n * (BLOB + PROOFS), "flops": n * PROOF_OPS}
    if kind == "cells_proofs":
        return {"bytes": n * (BLOB + CELLS + PROOFS), "flops": n * (PROOF_OPS + EXTEND_OPS)}
    if kind in ("recover", "recover_device"):
        return {"bytes": n * (CELLS + 128 + CELLS), "flops": n * RECOVER_OPS}
    if kind == "recover_proofs":
        return {"bytes": n * (CELLS + 128 + CELLS + PROOFS), "flops": n * (RECOVER_OPS + PROOF_OPS)}
    return {"bytes": n * (BLOB + 48), "flops": n * COMMIT_OPS}


def exact(case, seed):
    """Nothing here has a value in 64 bits: every output is bytes of whole numbers, or a verdict."""
    return None
