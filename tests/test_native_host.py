"""The native host path (csrc/fdb_torch.cpp): the mask-bounds kernel against padding.seq_bounds."""
import pytest
import torch

from flashdeberta_amd import _lib
from flashdeberta_amd.padding import key_padding_mask, seq_bounds


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bool, torch.uint8, torch.int32, torch.int64, torch.bfloat16, torch.float32, torch.float64])
@pytest.mark.parametrize("B,L", [(1, 1), (3, 40), (2, 255), (2, 257), (1, 1030)])
def test_mask_bounds(dtype, B, L):
    g = torch.Generator().manual_seed(L)
    rows = torch.zeros(B + 3, L)
    for b in range(B):
        lo = int(torch.randint(0, L, (1,), generator=g))
        rows[b, lo:int(torch.randint(lo, L, (1,), generator=g)) + 1] = 1
    rows[B + 1] = (torch.rand(L, generator=g) < 0.5).float()  # holes; row B stays empty
    rows[B + 2] = 1
    mask = rows.to(dtype).cuda()
    if dtype.is_floating_point:
        mask = torch.where(mask == 0, torch.full_like(mask, -0.0), mask)
    square = mask[:, None, None, :] * mask[:, None, :, None]
    for m in (mask, mask.t().contiguous().t(), square, square[:, 0]):
        start, length = _lib.native.mask_bounds(m)
        ref_start, ref_length, _ = seq_bounds(key_padding_mask(m))
        assert torch.equal(start, ref_start) and torch.equal(length, ref_length), (m.shape, start, ref_start, length, ref_length)
