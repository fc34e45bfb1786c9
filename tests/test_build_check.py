"""CPU test of the build's own check: no function of the device code that
returns to a caller is longer than a branch reaches."""
import pytest

from vkzg_amd import _lib
from vkzg_amd import build


def test_device_functions_are_within_a_branchs_reach():
    found = build.device_functions(_lib.LIB_PATH)
    for name in ("phase_a_slow", "phase_b_slow", "phase_b_slow_xyzz", "reduce_slow", "table_run_slow"):
        assert any(name in f for f in found), name  # the check sees them
    assert not any("k_bucket_reduce" in f or "k_pair_final" in f for f in found)  # kernels are not meant
    build.check_device_functions(_lib.LIB_PATH)


def test_a_longer_function_fails_the_build():
    size, name = max((b, f) for f, b in build.device_functions(_lib.LIB_PATH).items())
    with pytest.raises(RuntimeError, match="longer than a branch reaches.*" + name):
        build.check_device_functions(_lib.LIB_PATH, limit=size - 1)
