"""The fp32 forward with position terms at head_dim 64 (csrc/fdb_near_f32.hip): around its steps of 32 keys and tiles of 128 queries, far steps on
either side, shares of the keys, and rows that have no soft-max."""
import numpy as np
import pytest
import torch

from flashdeberta_amd import ops
from oracle import disentangled_oracle as O

pytestmark = pytest.mark.gpu

BOTH, C2P, P2C = (1, 1), (1, 0), (0, 1)


def _inputs(B, L, H, span, terms):
    g = torch.Generator().manual_seed(B * L)
    q, k, v = [torch.randn(B, L, H, 64, generator=g) for _ in range(3)]
    pk, pq = [torch.randn(H, 2 * span, 64, generator=g) if t else None for t in terms]
    return q, k, v, pk, pq


def _oracle(q, k, v, pk, pq, buckets, most, **kw):
    n = lambda x: None if x is None else x.numpy().astype(np.float64)
    t = lambda x: n(x).transpose(0, 2, 1, 3)
    out, lse = O.disentangled_attention(t(q), t(k), t(v), n(pk), n(pq), buckets, most, return_lse=True, **kw)
    return out.transpose(0, 2, 1, 3), lse.transpose(0, 2, 1)


@pytest.mark.parametrize("B,L,buckets,most,terms,causal,shares", [
    (2, 1, 32, 64, BOTH, False, 0), (1, 31, 32, 64, BOTH, False, 0), (1, 32, 256, 512, BOTH, False, 2), (1, 33, 32, 64, BOTH, True, 0),
    (1, 97, 32, 64, BOTH, False, 4), (1, 128, 256, 512, C2P, False, 0), (2, 129, 32, 64, P2C, False, 3),
    (1, 222, 32, 64, BOTH, False, 0), (1, 255, 0, 48, BOTH, True, 0), (1, 511, 32, 64, BOTH, False, 2), (1, 639, 256, 512, BOTH, False, 4),
    (1, 700, 32, 64, C2P, False, 1), (1, 705, 32, 64, P2C, True, 0), (1, 737, 256, 512, BOTH, False, 1), (1, 1300, 256, 512, BOTH, True, 0)])
def test_against_the_oracle(B, L, buckets, most, terms, causal, shares):
    q, k, v, pk, pq = x = _inputs(B, L, 2, ops.att_span(buckets, most), terms)
    ref, ref_lse = _oracle(*x, buckets, most, causal=causal)
    out, lse = ops.disentangled_attention_fwd(*[None if t is None else t.cuda() for t in x], position_buckets=buckets, max_relative_positions=most, causal=causal,
                                              return_lse=True, far_splits=shares)
    # scores are sums of at most 3 x 64 products of unit normal values: 2^-24 of sums up to about 40 each step, and the same again in the exponent
    assert np.abs(out.cpu().numpy() - ref).max() <= 2e-5 * max(1.0, np.abs(ref).max())
    assert np.abs(lse.view(B, L, 2).cpu().numpy() - ref_lse).max() <= 2e-5


@pytest.mark.parametrize("shares", [1, 2, 4])
def test_rows_without_a_soft_max(shares):
    """A query of NaN, one whose scores are all -inf, and keys whose scores are -inf for every query, a whole share of them."""
    q, k, v, pk, _ = _inputs(1, 300, 2, 32, C2P)
    pk[..., 0] = 0.0
    q[..., 0], k[..., 0] = 1.0, 0.0
    k[0, :160, :, 0] = -float("inf")
    q[0, 7] = float("nan")
    args = dict(position_buckets=32, max_relative_positions=64, far_splits=shares)
    call = lambda *x: ops.disentangled_attention_fwd(*[t.cuda() for t in x], None, return_lse=True, **args)
    out, lse = [t.cpu() for t in call(q, k, v, pk)]
    rows = [i for i in range(300) if i != 7]
    assert out[0, 7].isnan().all() and lse.view(300, 2)[7].isnan().all()
    assert out[0, rows].isfinite().all() and lse.view(300, 2)[rows].isfinite().all()
    seen = [t.clone() for t in (q, k, v)]
    seen[1][0, :160] = 5.0   # what these keys and values hold otherwise does not count
    seen[1][0, :160, :, 0] = -float("inf")
    seen[2][0, :160] = 3.0
    assert torch.equal(call(*seen, pk)[0].cpu()[0, rows], out[0, rows])
    k[0, :, :, 0] = -float("inf")
    out, lse = [t.cpu() for t in call(q, k, v, pk)]
    assert out.isnan().all() and lse.isnan().all()


@pytest.mark.parametrize("rise", [1, -1])
@pytest.mark.parametrize("L,terms,causal,shares", [(700, BOTH, False, 1), (641, C2P, False, 3), (993, P2C, False, 2), (900, BOTH, True, 0), (193, BOTH, False, 1)])
def test_scores_that_rise_through_the_far_steps(L, terms, causal, shares, rise):
    """A far step finds its reference point too low by the sum of its probabilities: scores that rise by 60 towards either end, by jumps and slowly."""
    q, k, v, pk, pq = x = _inputs(1, L, 2, 32, terms)
    j = torch.arange(L)
    height = (j if rise > 0 else L - 1 - j) / L
    q[..., 0], k[..., 0] = 3.0, (torch.where(j % 64 < 32, height, (height * 6).floor() / 6) * 20.0 * (64.0 * (1 + sum(terms))) ** 0.5)[None, :, None]
    q[0, 5] = 0.0   # a row that sees none of it
    for t in (pk, pq):
        if t is not None:
            t[..., 0] = 0.0
    ref, ref_lse = _oracle(*x, 32, 64, causal=causal)
    out, lse = ops.disentangled_attention_fwd(*[None if t is None else t.cuda() for t in x], position_buckets=32, max_relative_positions=64, causal=causal, return_lse=True,
                                              far_splits=shares)
    # a score of 60 carries 2^-24 of itself from each of some ten sums that are as large: 4e-5 of a probability, and as much of lse
    assert np.abs(out.cpu().numpy() - ref).max() <= 1e-4 * max(1.0, np.abs(ref).max())
    assert np.abs(lse.view(1, L, 2).cpu().numpy() - ref_lse).max() <= 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,H,padded", [(1, 1, 1, False), (3, 70, 7, True), (700, 3, 5, False), (2800, 129, 12, True)])   # the last: past 2^22 rows of the outputs
def test_merged_shares_lie_where_one_launch_puts_them(B, L, H, padded):
    g = torch.Generator(device="cuda").manual_seed(B + L)
    q, k, v = [torch.randn(B, L, H, 64, device="cuda", generator=g) for _ in range(3)]
    pk, pq = [torch.randn(H, 64, 64, device="cuda", generator=g) for _ in range(2)]
    kw = dict(position_buckets=32, max_relative_positions=64, return_lse=True)
    if padded:
        kw["seq_len"] = torch.randint(0, L + 1, (B,), device="cuda", generator=g, dtype=torch.int32)
    (one, one_lse), (shared, shared_lse) = [ops.disentangled_attention_fwd(q, k, v, pk, pq, far_splits=n, **kw) for n in (1, 2)]
    # sums in another order: a few 2^-24 of outputs whose weights are at most 1, and of log-sum-exps of at most 40
    assert (shared - one).abs().max() <= 4e-6 * max(1.0, one.abs().max().item()) and (shared_lse - one_lse).nan_to_num(posinf=0, neginf=0).abs().max() <= 1e-5
    assert torch.equal(shared_lse.isinf(), one_lse.isinf())
