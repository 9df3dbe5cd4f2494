"""Registers that the compiler gave kernels whose speed is how many waves a SIMD holds, or whose registers are full (tests/code_objects.py; without a GPU)."""
import pytest

from code_objects import kernels
from flashdeberta_amd import _lib


@pytest.fixture(scope="module")
def built():
    return kernels(_lib.LIB_PATH)


def test_merges_hold_eight_waves_a_simd(built):
    merges = {name: k[".vgpr_count"] for name, k in built.items() if "fdb_merge_" in name}
    assert len(merges) == 2 + 9 and max(merges.values()) <= 64, merges
