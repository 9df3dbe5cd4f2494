"""The packed layout's work-list (csrc/fdb_aux.hip) where its threads share out sequences and pairs unevenly."""
import numpy as np
import pytest
import torch

from flashdeberta_amd import _lib


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 15, 16, 17, 63, 64, 65, 1023, 1024, 1025, 2100])
def test_every_tile_once_and_in_order(batch):
    rng = np.random.default_rng(batch)
    lens = rng.integers(0, 400, size=batch)
    lens[::3] = 128                                                                # ties, whole tiles
    lens[batch // 2], lens[-1] = 128 * 16 + 1, 128 * 33 if batch % 2 else 0        # more tiles than threads, empty at the end
    cu = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).cuda()
    total = int(lens.sum())
    ints = int(_lib.lib.fdb_worklist_ints(total, batch))
    wl = torch.full((ints + 4,), -7, dtype=torch.int32, device="cuda")
    assert _lib.lib.fdb_build_worklist(cu.data_ptr(), batch, total, wl.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    got = wl.cpu().numpy()
    order = sorted(range(batch), key=lambda b: (-int(lens[b]), b)) if batch <= 1024 else range(batch)
    want = [[b, m0] for b in order for m0 in range(0, int(lens[b]), 128)]
    assert got[0] == len(want) and got[1] == 0
    assert got[2:2 + 2 * len(want)].reshape(-1, 2).tolist() == want
    assert (got[2 + 2 * len(want):] == -7).all()
