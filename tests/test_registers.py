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


def _one_kernel(built, name, c2p, p2c):
    """The kernel for both launches in one, head_dim 128"""
    return next(k for n, k in built.items() if "fdb_attn_kernelIN3fdb%sES2_Li128ELb0ELb%dELb%dELi0E" % (name, c2p, p2c) in n)


@pytest.mark.parametrize("name", ["6Bf16Tr", "5F16Tr"], ids=["bf16", "fp16"])
def test_full_registers_take_no_arguments_ahead(built, name):
    """Bytes of scratch a lane at head_dim 128, where two workgroups a compute unit leave 256 registers: what is read ahead is spilled for.  bf16 with c2p alone
    is the one whose 12 bytes more came with fewer spills."""
    most = {(0, 0): 84, (0, 1): 52, (1, 0): 124 if name == "6Bf16Tr" else 108, (1, 1): 0}
    got = {terms: _one_kernel(built, name, *terms)[".private_segment_fixed_size"] for terms in most}
    assert all(got[terms] <= most[terms] for terms in most), got


def test_the_e4m3_far_launch_keeps_its_scalars(built):
    """Three workgroups a compute unit: with the arguments read ahead 20 scalar registers were spilled."""
    far = {n: k[".sgpr_spill_count"] for n, k in built.items() if "fdb_far8_kernel" in n}
    assert len(far) == 3 and max(far.values()) <= 4, far


def test_products_of_real_rows_hold_no_bias_through_the_tile(built):
    """172 registers, 188 with what the end of the tile reads asked for ahead, which made these products slower."""
    real = [k[".vgpr_count"] for n, k in built.items() if "fdb_gemm_real_kernel" in n]
    assert len(real) == 2 and max(real) <= 176, real
