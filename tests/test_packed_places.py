"""Packed batches of up to 64 sequences, whose workgroups find their query tiles without a work-list (packed_place in csrc/fdb_device.h): the bits of the same
sequences in a batch of more than 64, which has one."""
import random

import pytest
import torch

from flashdeberta_amd import _lib, ops


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "fp32", "e4m3", "head_dim 32", "one kernel"])
@pytest.mark.parametrize("batch,longest,heads", [(1, 1, 48), (1, 700, 48), (2, 128, 48), (7, 250, 48), (6, 500, 48), (63, 300, 4), (64, 40, 8), (64, 500, 3)])
def test_bits_of_the_work_list(batch, longest, heads, kind):
    rng = random.Random(batch + longest)
    lens = [rng.choice([0, 1, 127, 128, 129, 256, rng.randint(0, longest)]) % (longest + 1) for _ in range(batch - 1)] + [longest]
    rng.shuffle(lens)
    H, D, T = heads, 32 if kind == "head_dim 32" else 64, sum(lens)
    dtype = torch.float32 if kind == "fp32" else torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(T)
    q, k, v = [torch.randn(T, H, D, device="cuda", generator=g).to(dtype) for _ in range(3)]
    pk, pq = [torch.randn(H, 64, D, device="cuda", generator=g).to(dtype) for _ in range(2)]
    kw = dict(max_seqlen=longest, position_buckets=32, max_relative_positions=64, single_kernel=kind == "one kernel", far_splits=1)
    if kind not in ("one kernel", "head_dim 32", "fp32"):
        kw["near_splits"] = 1   # as many shares whatever the batch; so many heads that no workgroup is two teams in one of the two
    if kind == "e4m3":
        q, kw["q_scale"], k, kw["k_scale"] = ops.quantize_e4m3_per_head_pair(q, k)
        (pk, kw["pos_key_scale"]), (pq, kw["pos_query_scale"]) = [(y.transpose(0, 1), z) for y, z in (ops.quantize_e4m3_per_head(t.transpose(0, 1)) for t in (pk, pq))]
    needs = _lib.lib.fdb_needs_worklist
    assert not needs(T, batch, H) and needs(T, batch + 65, H)
    got = []
    for empty in (0, 65):
        ends = torch.tensor([0] + lens + [0] * empty, dtype=torch.int32).cumsum(0, dtype=torch.int32).cuda()
        out = torch.full((T, H, D), 7.0, device="cuda", dtype=v.dtype)
        got.append(ops.disentangled_attention_fwd(q, k, v, pk, pq, cu_seqlens=ends, out=out, **kw))
    assert torch.equal(*got)
