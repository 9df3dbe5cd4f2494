"""Padded batches whose workgroups are dealt by the lengths of their sequences (padded_map in csrc/fdb_device.h): the bits of the same sequences in a batch of more
than 64, which is dealt in the plain order."""
import random

import pytest
import torch

from flashdeberta_amd import ops

pytestmark = pytest.mark.gpu


def _bounds(kind, B, L):
    rng = random.Random(B * 1000 + L)
    starts = [0] * B
    if kind == "ragged":
        lens = [rng.randint(0, L) for _ in range(B)]
    elif kind == "equal":
        lens = [L // 2] * B
    elif kind == "left":
        lens = [rng.randint(1, L) for _ in range(B)]
        starts = [L - n for n in lens]
    else:   # what bounds may hold: none, a row that cannot be expressed, past the end, a start and a length past the end
        lens = [rng.choice([0, -1, L, L + 7, 1, 128, 129]) for _ in range(B)]
        starts = [rng.choice([0, 0, -3, L - 1, L + 2]) for _ in range(B)]
    return starts, lens


def _call(x, starts, lens, more, grads):
    """Forward (and backward) of the batch and, `more`, as many empty sequences behind it."""
    q, k, v, pk, pq, dout = x
    wide = lambda t: torch.cat([t, torch.zeros(more, *t.shape[1:], device="cuda", dtype=t.dtype)]) if more else t
    vec = lambda t: torch.tensor(list(t) + [0] * more, dtype=torch.int32, device="cuda")
    kw = dict(position_buckets=32, max_relative_positions=64, seq_start=vec(starts) if any(starts) else None, seq_len=vec(lens))
    q, k, v, dout = [wide(t) for t in (q, k, v, dout)]
    hold = torch.full((q.numel() * 4,), float("nan"), device="cuda", dtype=q.dtype)
    del hold   # what the outputs are given
    out, lse = ops.disentangled_attention_fwd(q, k, v, pk, pq, return_lse=True, **kw)
    n = out.shape[0] - more
    res = [out[:n], lse.view(out.shape[0], -1)[:n]]
    if grads:
        res += [g[:n] for g in ops.disentangled_attention_bwd(q, k, v, out, lse, dout, pk, pq, **kw)[:3]]
    return [t.nan_to_num(nan=12345.0) for t in res]


@pytest.mark.parametrize("kind", ["ragged", "equal", "left", "odd"])
@pytest.mark.parametrize("B,L,H,dtype", [(2, 600, 32, torch.bfloat16), (64, 130, 3, torch.float16), (33, 129, 5, torch.bfloat16), (23, 385, 4, torch.bfloat16), (9, 1100, 6, torch.float16),
                                         (40, 200, 4, torch.float32), (64, 520, 8, torch.bfloat16)])   # the last: the backward's roles as two launches
def test_bits_of_the_plain_order(B, L, H, dtype, kind):
    g = torch.Generator(device="cuda").manual_seed(B + L)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)
    x = rnd(B, L, H, 64), rnd(B, L, H, 64), rnd(B, L, H, 64), rnd(H, 64, 64), rnd(H, 64, 64), rnd(B, L, H, 64)
    starts, lens = _bounds(kind, B, L)
    assert B * ((L + 127) // 128) * H > 256
    grads = dtype != torch.float32 and min(lens) >= 0
    for a, b in zip(_call(x, starts, lens, 0, grads), _call(x, starts, lens, 65, grads)):
        assert torch.equal(a, b)
