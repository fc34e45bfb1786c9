"""CPU tests of the library's host code: libvkzg.so in a process of its own
against tests/c/hip_host.cpp, a HIP runtime whose device memory is host memory
and whose kernels are only counted.  What is checked is what the host decides:
what a call does after one that failed, which plan it takes, what it counts."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)

PREAMBLE = """
import ctypes, os, sys
H = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
for f in ("host_live", "host_launches", "host_copies"):
    getattr(H, f).restype = ctypes.c_uint64
H.host_fail_alloc.argtypes = [ctypes.c_int64]
H.host_fail_left.restype = ctypes.c_int64
H.host_limit.argtypes = [ctypes.c_uint64]
sys.path.insert(0, sys.argv[2])
import vkzg_amd
BLOB, CELLS, GIB = 131072, 262144, 1 << 30

def launches(name):
    return H.host_launches(name.encode())
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip") / "hip_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", so, os.path.join(HERE, "c", "hip_host.cpp")], check=True)

    def script(body, **env):
        r = subprocess.run([sys.executable, "-c", PREAMBLE + body, so, REPO], capture_output=True, text=True,
                           timeout=100, env=dict(os.environ, VKZG_AMD_WINDOW="6", **env))
        assert r.returncode == 0, r.stdout + r.stderr

    return script


def test_commitments_after_an_allocation_that_failed(run):
    """Whichever allocation of a prover's first commitment call fails, the call
    either reports it or takes the bucket method, and the next one is summed from
    a table that was built whole: never from one that a failure cut short."""
    run("""
def table_build(p):
    before = launches("k_table_multiples"), launches("k_phase_a"), launches("k_msm_buckets")
    try:
        p.blob_to_kzg_commitments(bytes(BLOB), 1)
        ok = True
    except vkzg_amd.VkzgError:
        ok = False
    after = launches("k_table_multiples"), launches("k_phase_a"), launches("k_msm_buckets")
    return (ok,) + tuple(b - a for a, b in zip(before, after))

with vkzg_amd.Prover(max_batch_size=1) as p:
    first = table_build(p)
    whole, live = first[1], H.host_live()
    assert first[0] and whole > 1 and first[2] == 1 and table_build(p) == (True, 0, 1, 0)
k = 0
while True:
    k += 1
    with vkzg_amd.Prover(max_batch_size=1) as p:
        H.host_fail_alloc(k)
        one = table_build(p)
        if H.host_fail_left() > 0:
            break  # the call makes fewer allocations than that
        H.host_fail_alloc(0)
        if one[0] and one[1] < whole:
            assert one[2] == 0 and one[3] == 1, (k, one)  # no table: buckets
        two, three = table_build(p), table_build(p)
        assert two[0] and two[2] == 1 and sorted((one[1], two[1])) == [0, whole], (k, one, two)
        assert three == (True, 0, 1, 0), (k, three)
        assert abs(H.host_live() - live) < 8 << 20, (k, H.host_live() - live)  # nothing of the failed build is kept
H.host_fail_alloc(0)
assert k > 6 and H.host_live() == 0
""")


@pytest.mark.parametrize("free_gib,windows", [(200, 25), (32, 28), (20, 31), (10, 36), (3, 63), (1.2, 127), (0.5, 0), (0.01, 0)])
def test_commitment_plan_fits_the_free_memory(run, free_gib, windows):
    """The first commitment call within the free memory there is, temporaries
    included: fewer windows' larger tables while there is plenty, the bucket
    method where no table fits."""
    run("""
free, windows = %r, %d
with vkzg_amd.Prover(max_batch_size=1) as p:
    H.host_limit(int(H.host_live() + free * GIB))
    before = H.host_live()
    p.blob_to_kzg_commitments(bytes(2 * BLOB), 2)
    held = H.host_live() - before
    if windows == 0:
        assert launches("k_msm_buckets") > 0 and launches("k_phase_a") == 0 and held < free * GIB / 2
    else:
        c, k = 255 // windows, 255 %% windows
        table = 4096 * (windows + k) * 2 ** (c - 1) * 128
        assert launches("k_msm_buckets") == 0 and table <= held < table + (16 << 20) and table <= free * GIB / 8
    p.blob_to_kzg_commitments(bytes(65 * BLOB), 65)
""" % (free_gib, windows))


def test_a_tuning_can_be_put_back(run):
    """Fields that are fitted to each batch are fitted again, at every size of the
    class, after a tuning that get_tuning reported is set: straight away, after a
    change in between, and after one that touched another field only.  What is set
    is what get_tuning reports for that size."""
    run("""
classes = [(1,), range(2, 5), range(5, 17), range(17, 65), (65, 100, 200, 256)]
with vkzg_amd.Prover(max_batch_size=256) as p:
    want = {n: p.get_tuning(n) for c in classes for n in c}
    assert len({(t["phase_a_groups"], t["reduce_lanes"]) for t in want.values()}) > 4  # the fits do vary
    for c in classes:
        for n in c:
            saved = p.get_tuning(n)
            p.set_tuning(n, **saved)
            assert all(p.get_tuning(m) == want[m] for m in c), n
            for change in (dict(phase_a_groups=3), dict(reduce_lanes=8, phase_a_groups=20, ladder_splits=4),
                           dict(ladder_splits=2), dict(splits=2), dict(phase_a_groups=7, splits=3)):
                p.set_tuning(n, **change)
                assert p.get_tuning(n) == dict(saved, **change), (n, change)
                p.set_tuning(n, **saved)
                assert all(p.get_tuning(m) == want[m] for m in c), (n, change)
    p.set_tuning(11, splits=2)
    assert all(p.get_tuning(m) == dict(want[m], splits=2) for m in classes[2])
    for bad in (dict(phase_a_groups=0), dict(reduce_lanes=0), dict(phase_a_groups=21)):
        try:
            p.set_tuning(3, **bad)
            assert False, bad
        except vkzg_amd.VkzgError as e:
            assert e.code == vkzg_amd.ERR_BADARGS
    p.autotune()  # its choices are pinned, and stay so
    tuned = {n: p.get_tuning(n) for c in classes for n in c}
    assert sum(len({tuned[n]["phase_a_groups"] for n in c}) == 1 for c in classes[1:]) > 0
    assert sum(len({tuned[n]["reduce_lanes"] for n in c}) == 1 for c in classes[1:]) > 0
    for n in (1, 3, 11, 40, 200):
        p.set_tuning(n, phase_a_groups=9)
        p.set_tuning(n, **tuned[n])
    assert all(p.get_tuning(n) == t for n, t in tuned.items())
""")


def test_resident_tables_count_the_commitments_table(run):
    run("""
with vkzg_amd.Prover(max_batch_size=1) as p:
    one = p.info()["resident_table_bytes"]
    vkzg_amd.Server(p, batch_blobs=1, slots=1, hbm_budget_bytes=one + (64 << 20)).close()
    before = H.host_live()
    p.blob_to_kzg_commitments(bytes(BLOB), 1)
    two = p.info()["resident_table_bytes"]
    table = 4096 * 30 * 512 * 128  # 25 windows, 5 of them a bit wider
    assert two - one == table and table <= H.host_live() - before < table + (32 << 20)
    for budget in (one + (64 << 20), two):
        try:
            vkzg_amd.Server(p, batch_blobs=1, slots=1, hbm_budget_bytes=budget)
            assert False, budget
        except vkzg_amd.VkzgError as e:
            assert e.code == vkzg_amd.ERR_MALLOC
    vkzg_amd.Server(p, batch_blobs=1, slots=1, hbm_budget_bytes=two + (64 << 20)).close()
""")


def test_a_servers_slots_stay_within_its_budget(run):
    """What a server allocates is what its budget leaves beside the tables, with
    slots of one blob and of many; the prover reports its own working set whole."""
    run("""
for n in (1, 2, 7, 8, 20):
    before = H.host_live()
    with vkzg_amd.Prover(max_batch_size=n) as p:
        info = p.info()
        took = H.host_live() - before - info["resident_table_bytes"]
        assert 0 <= took - info["working_bytes"] < 4 << 20, (n, took, info)  # the setup's points, roots and items
with vkzg_amd.Prover(max_batch_size=20) as p:
    tables = p.info()["resident_table_bytes"]
    with vkzg_amd.Server(p, batch_blobs=1, slots=1) as s:
        per_blob = s.stats()["slot_bytes"]
    for blobs, slots in ((1, 1), (1, 4), (3, 2), (7, 1), (8, 2), (64, 3)):
        for room in (1.0, 1.5, 2.0, 4.2, 9.9, 30.0):
            budget = tables + int(per_blob * room)
            before = H.host_live()
            with vkzg_amd.Server(p, batch_blobs=blobs, slots=slots, hbm_budget_bytes=budget) as s:
                st = s.stats()
                took = H.host_live() - before
                assert took <= budget - tables, (blobs, slots, room, took)
                assert st["slots"] * st["slot_bytes"] <= took <= st["slots"] * (st["slot_bytes"] + (16 << 20))
                assert st["batch_blobs"] == min(blobs, int(room))
""")


def test_every_size_of_a_call_keeps_its_graphs(run):
    """Cells with proofs at every batch size up to 160, again and again: captured
    the first time only, though each call is two graphs."""
    run("""
L = vkzg_amd._lib.load()
n = 160
blobs, cells, proofs = (ctypes.create_string_buffer(n * k) for k in (BLOB, CELLS, 128 * 48))
with vkzg_amd.Prover(max_batch_size=n) as p:
    for rep in range(2):
        for k in range(1, n + 1):
            assert L.vkzg_amd_compute_cells_and_proofs(p.handle, cells, proofs, blobs, k) == 0
    assert p.info()["graph_captures"] == 2 * n and p.info()["graph_replays"] == 2 * n
""")


def test_large_copies_are_few(run):
    """A copy of up to 12 MiB takes at most three DMAs each way: with more, calls on
    buffers in use are slower than with one."""
    run("""
L = vkzg_amd._lib.load()
n = 97
cells, out = ctypes.create_string_buffer(n * CELLS), ctypes.create_string_buffer(n * CELLS)
mask = ctypes.create_string_buffer(bytes([1] * 64 + [0] * 64) * n, n * 128)
with vkzg_amd.Prover(max_batch_size=n) as p:
    for k in list(range(1, 50)) + [96, 97]:
        before = H.host_copies()
        assert L.vkzg_recover_cells_batch(p.handle, out, cells, mask, k) == 0
        dmas = H.host_copies() - before
        assert dmas == 0 if k < 12 else dmas <= 6 if k <= 48 else dmas <= 2 * -(-k * CELLS // (4 << 20)), (k, dmas)
""")
