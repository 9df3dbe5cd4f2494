"""The near launch with all key tiles, taken where a far launch would have little to do: against the oracle, around the tile edges, and
against the pair of launches, which far_splits=1 asks for."""
import ctypes

import numpy as np
import pytest
import torch

from flashdeberta_amd import _lib, ops
from launches import launches
from oracle import disentangled_oracle as O
from test_launches import _forward

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _inputs(B, L, H, terms, dtype):
    g = torch.Generator().manual_seed(B * L)
    q, k, v = [torch.randn(B, L, H, 64, generator=g).to(dtype) for _ in range(3)]
    pk, pq = [torch.randn(H, 512, 64, generator=g).to(dtype) if t else None for t in terms]
    return q, k, v, pk, pq


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("B,L,terms", [(1, 577, (1, 1)), (1, 640, (1, 1)), (2, 641, (1, 0)), (1, 777, (0, 1)), (1, 1024, (1, 1)), (1, 1153, (1, 1))])
def test_all_key_tiles_in_the_near_launch(B, L, terms, dtype):
    q, k, v, pk, pq = _inputs(B, L, 2, terms, dtype)
    n = lambda x: None if x is None else x.float().numpy().astype(np.float64)
    t = lambda x: n(x).transpose(0, 2, 1, 3)
    ref, ref_lse = O.disentangled_attention(t(q), t(k), t(v), n(pk), n(pq), 256, 512, return_lse=True)
    d = lambda x: None if x is None else x.cuda()
    kw = dict(position_buckets=256, max_relative_positions=512, return_lse=True)
    out, lse = ops.disentangled_attention_fwd(d(q), d(k), d(v), d(pk), d(pq), **kw)
    two, two_lse = ops.disentangled_attention_fwd(d(q), d(k), d(v), d(pk), d(pq), far_splits=1, **kw)
    # scores of standard deviation 1.0 to 1.4 carry a rounding of the scaled query and of c2p, the output a rounding of the probabilities and one of its own
    for got, got_lse in ((out, lse), (two, two_lse)):
        assert np.abs(got.float().cpu().numpy().transpose(0, 2, 1, 3) - ref).max() <= 3 * EPS[dtype] * max(1.0, np.abs(ref).max())
        assert np.abs(got_lse.view(B, L, 2).cpu().numpy().transpose(0, 2, 1) - ref_lse).max() <= 2 * EPS[dtype]


@pytest.mark.gpu
def test_padded_rows_in_the_near_launch():
    q, k, v, pk, pq = [x.cuda() for x in _inputs(3, 777, 2, (1, 1), torch.bfloat16)]
    kw = dict(position_buckets=256, max_relative_positions=512)
    start, length = [torch.tensor(x, dtype=torch.int32, device="cuda") for x in ((0, 100, 776), (777, 640, 1))]
    out = ops.disentangled_attention_fwd(q, k, v, pk, pq, seq_start=start, seq_len=length, **kw)
    for b in range(3):
        s, n = int(start[b]), int(length[b])
        alone = ops.disentangled_attention_fwd(*[x[b:b + 1, s:s + n].contiguous() for x in (q, k, v)], pk, pq, far_splits=1, **kw)
        assert (out[b, s:s + n] - alone[0]).abs().max() <= 4 * EPS[torch.bfloat16]
        assert out[b].isfinite().all() and (out[b, :s] == 0).all() and (out[b, s + n:] == 0).all()


def test_workspace_of_a_far_share():
    """A far share of its own has a workspace slot: none is asked for where the near launch takes all, whatever the number of near shares."""
    a = _lib.FdbAttnArgs()
    for n in ("q", "k", "v", "out", "pos_key", "pos_query", "lse", "delta_lut"):
        setattr(a, n, 0x1000)
    a.batch, a.heads, a.head_dim, a.dtype, a.att_span, a.lut_radius, a.max_seqlen, a.total_tokens = 1, 1, 64, _lib.FDB_BF16, 256, 512, 2048, 2048
    part = lambda rows: rows * (64 * 2 + 4)
    ws = lambda: _lib.lib.fdb_attn_workspace_bytes(ctypes.byref(a))
    assert ws() % part(2048) == 0
    near = ws() // part(2048)
    a.far_splits = 2
    assert ws() == (1 + near) * part(2048)


def _errors(B, L, H, kind, buckets=256, most=512, **kw):
    """Errors of the output [L, H, 64] and of the log-sum-exp [L, H], first batch row, against 64 bits on the operands as the kernels get them."""
    q, k, v, pk, pq = _inputs(B, L, H, (1, 1), torch.float16 if kind == "fp16" else torch.bfloat16)
    pk, pq = pk[:, :2 * buckets], pq[:, :2 * buckets]
    call, given = dict(position_buckets=buckets, max_relative_positions=most, return_lse=True, **kw), [x.cuda() for x in (q, k, v, pk, pq)]
    exact = [x.double() for x in (q, k, v, pk, pq)]
    if kind == "e4m3":
        eight = [ops.quantize_e4m3_per_head(x) for x in (given[0].view(B * L, H, 64), given[1].view(B * L, H, 64), given[3].transpose(0, 1), given[4].transpose(0, 1))]
        plain = [y.double().cpu() * s.double().cpu()[:, None] for y, s in eight]
        exact = [plain[0].view(B, L, H, 64), plain[1].view(B, L, H, 64), exact[2], plain[2].transpose(0, 1), plain[3].transpose(0, 1)]
        (q8, qs), (k8, ks), (pk8, pks), (pq8, pqs) = eight
        given = [q8.view(B, L, H, 64), k8.view(B, L, H, 64), given[2], pk8.transpose(0, 1), pq8.transpose(0, 1)]
        call.update(q_scale=qs, k_scale=ks, pos_key_scale=pks, pos_query_scale=pqs)
    rows = lambda x: x[:1].numpy().transpose(0, 2, 1, 3)
    ref, ref_lse = O.disentangled_attention(*[rows(x) for x in exact[:3]], exact[3].numpy(), exact[4].numpy(), buckets, most, return_lse=True)
    out, lse = ops.disentangled_attention_fwd(*given, **call)
    e = out[0].double().cpu().numpy() - ref[0].transpose(1, 0, 2)
    return e, lse.view(B, L, H)[0].double().cpu().numpy() - ref_lse[0].T


def _rms(*args, **kw):
    """... their root mean squares, and that of the log-sum-exp of the two rows at either end"""
    e, el = _errors(*args, **kw)
    return np.sqrt((e * e).mean()), np.sqrt((el * el).mean()), np.sqrt((el[[0, 1, -2, -1]] ** 2).mean())


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "fp16", "e4m3"])
@pytest.mark.parametrize("B,L,H", [(3, 777, 12), (2, 1024, 12), (1, 1300, 12), (1, 2000, 4)])
def test_no_less_precise_than_two_launches(B, L, H, kind):
    """What a row has in common with all far keys of a side goes whole into its log-sum-exp: rounded to 16 bits it made the error up to 2.6 times as large."""
    one, two = _rms(B, L, H, kind), _rms(B, L, H, kind, far_splits=1)
    # root mean squares over 9000 rows: two samples of one error differ by about a hundredth
    assert one[0] <= 1.03 * two[0] and one[1] <= 1.03 * two[1], (one, two)


@pytest.mark.gpu
def test_e4m3_far_keys_add_nothing_to_the_rounding_of_c2p():
    """In e4m3 the near steps' c2p is cut to 16 bits, the far ones' is not: at the ends of 1500 tokens, where 700 at most are near, the log-sum-exp's
    error is that share (and less) of a call's whose keys are all near."""
    assert _rms(1, 1500, 4, "e4m3")[2] <= 700 / 1500 * 1.25 * _rms(1, 512, 12, "e4m3")[2]   # 32 rows: a root mean square known to a quarter


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "fp16", "e4m3"])
@pytest.mark.parametrize("shared", [True, False])
# all near but one key; ragged last steps that are near and far ones; shares that hold no near step, far ones of either side or of both; the most tiles
@pytest.mark.parametrize("L,H,buckets,most", [(577, 3, 256, 512), (193, 2, 32, 64), (641, 1, 32, 64), (833, 2, 32, 64), (960, 12, 32, 64), (1000, 1, 128, 256),
                                              (2048, 2, 256, 512), (1985, 12, 256, 512)])
def test_far_steps_and_shares(L, H, buckets, most, shared, kind):
    e, el = _errors(1, L, H, kind, buckets, most, **({} if shared else dict(workspace=torch.empty(256, dtype=torch.uint8, device="cuda"))))
    eps = EPS[torch.float16 if kind == "fp16" else torch.bfloat16]
    # as above; outputs are of magnitude 1 at most at these lengths, and e4m3's near c2p is cut to fp16: a score of 4 by 2^-9
    assert np.abs(e).max() <= 3 * eps and np.abs(el).max() <= 2 * eps


@pytest.mark.gpu
@pytest.mark.parametrize("B,H", [(1, 1), (3, 7), (400001, 12)])   # the last: more workgroups than quick_div's fp32 quotients reach
def test_every_workgroup_finds_its_place(B, H):
    """Texts of one token: the output is v."""
    g = torch.Generator(device="cuda").manual_seed(B)
    q, k, v = [torch.randn(B, 1, H, 64, device="cuda", generator=g, dtype=torch.bfloat16) for _ in range(3)]
    pk, pq = [torch.randn(H, 64, 64, device="cuda", generator=g, dtype=torch.bfloat16) for _ in range(2)]
    assert torch.equal(ops.disentangled_attention_fwd(q, k, v, pk, pq, position_buckets=32, max_relative_positions=64), v)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("causal", [False, True], ids=["all", "causal"])
@pytest.mark.parametrize("L,terms,buckets,most", [(289, (1, 1), 32, 64), (320, (1, 0), 256, 512), (321, (0, 1), 32, 64), (352, (1, 1), 256, 512), (900, (1, 1), 32, 64)])
def test_two_teams(L, terms, buckets, most, causal, dtype):
    """Workgroups of two teams at even and odd numbers of steps, far ones among them, in padded rows down to no step for a team or for both, and the same sequences packed,
    whose mean length makes two teams at 900 alone."""
    lens = [L, 1, 33, 0, 64, L - 1]
    q, k, v, pk, pq = _inputs(len(lens), L, 2, terms, dtype)
    pk, pq = [None if x is None else x[:, :2 * buckets] for x in (pk, pq)]
    d = lambda x: None if x is None else x.cuda()
    kw = dict(position_buckets=buckets, max_relative_positions=most, causal=causal, return_lse=True)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    out, lse = ops.disentangled_attention_fwd(d(q), d(k), d(v), d(pk), d(pq), seq_len=i32(lens), **kw)
    rows = lambda x: torch.cat([x[b, :m] for b, m in enumerate(lens)])
    packed, packed_lse = ops.disentangled_attention_fwd(*[d(rows(x)) for x in (q, k, v)], d(pk), d(pq), cu_seqlens=i32(np.cumsum([0] + lens)), max_seqlen=L, **kw)
    lse = lse.view(len(lens), L, 2)
    assert torch.equal(out[:, L - 1:][[1, 2, 3, 4]], torch.zeros_like(out[:4, :1])) and (out[3] == 0).all()
    n = lambda x: None if x is None else x.float().numpy().astype(np.float64)
    at = 0
    for b, m in enumerate(lens):
        if m == 0:
            continue
        t = lambda x: n(x[b:b + 1, :m]).transpose(0, 2, 1, 3)
        ref, ref_lse = O.disentangled_attention(t(q), t(k), t(v), n(pk), n(pq), buckets, most, causal=causal, return_lse=True)
        ref, ref_lse = ref[0].transpose(1, 0, 2), ref_lse[0].T
        for got, got_lse in ((out[b, :m], lse[b, :m]), (packed[at:at + m], packed_lse.view(-1, 2)[at:at + m])):
            # scores and probabilities are rounded as in every near launch, see above
            assert np.abs(got.float().cpu().numpy() - ref).max() <= 3 * EPS[dtype] * max(1.0, np.abs(ref).max()), (b, m)
            assert np.abs(got_lse.cpu().numpy() - ref_lse).max() <= 2 * EPS[dtype], (b, m)
        at += m


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("causal", [False, True], ids=["all", "causal"])
@pytest.mark.parametrize("many", [False, True], ids=["few", "with a work-list"])
@pytest.mark.parametrize("L,terms,buckets,most", [(352, (1, 1), 256, 512), (353, (1, 0), 32, 64), (353, (0, 1), 256, 512), (384, (1, 1), 32, 64), (380, (0, 1), 32, 64)])
def test_two_teams_of_packed_sequences(L, terms, buckets, most, many, causal, dtype):
    """Two teams go by the mean length: 10 to 12 steps here, of sequences down to no token; up to 64 without a work-list, more with one."""
    lens, H = ([L] * 60 + [1, 33, 0, 64, 129, L - 1], 1) if many else ([L] * 16 + [1, 33, 0, 64, L - 1], 2)
    np.random.default_rng(L).shuffle(lens)
    T, i32 = sum(lens), lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    assert _lib.lib.fdb_needs_worklist(T, len(lens), H) == many
    (rc, made), = launches([_forward(len(lens), L, H, _lib.FDB_BF16, most, total_tokens=T, cu_seqlens=0x1000, worklist=0x1000, causal=int(causal))])
    assert rc == 0 and [m[2:] for m in made if "near" in m[0]] == [(1, 512)], made   # 512 threads: both teams
    q, k, v, pk, pq = _inputs(1, T, H, terms, dtype)
    pk, pq = [None if x is None else x[:, :2 * buckets] for x in (pk, pq)]
    d = lambda x: None if x is None else x.cuda()
    out, lse = ops.disentangled_attention_fwd(d(q[0]), d(k[0]), d(v[0]), d(pk), d(pq), cu_seqlens=i32(np.cumsum([0] + lens)), max_seqlen=L, position_buckets=buckets,
                                              max_relative_positions=most, causal=causal, return_lse=True, workspace=torch.empty(16, dtype=torch.uint8, device="cuda"))
    n = lambda x: None if x is None else x.float().numpy().astype(np.float64)
    at = 0
    for m in lens:
        if m == 0:
            continue
        t = lambda x: n(x[:, at:at + m]).transpose(0, 2, 1, 3)
        ref, ref_lse = O.disentangled_attention(t(q), t(k), t(v), n(pk), n(pq), buckets, most, causal=causal, return_lse=True)
        # scores and probabilities are rounded as in every near launch, see above
        assert np.abs(out[at:at + m].float().cpu().numpy() - ref[0].transpose(1, 0, 2)).max() <= 3 * EPS[dtype] * max(1.0, np.abs(ref).max()), (at, m)
        assert np.abs(lse.view(-1, H)[at:at + m].cpu().numpy() - ref_lse[0].T).max() <= 2 * EPS[dtype], (at, m)
        at += m


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("B,L,H,padded,far,near", [(1, 1, 1, False, 1, 2), (3, 70, 7, True, 1, 4), (700, 3, 5, False, 1, 3), (2, 700, 3, False, 2, 2), (2, 700, 3, True, 3, 2),
                                                   (2, 700, 3, True, 4, 4), (2800, 129, 12, True, 1, 2)])   # the last: past 2^22 rows of the outputs
def test_merged_shares_lie_where_one_launch_puts_them(B, L, H, padded, far, near, dtype):
    """Two to eight partial results of a row."""
    g = torch.Generator(device="cuda").manual_seed(B + L)
    q, k, v = [torch.randn(B, L, H, 64, device="cuda", generator=g, dtype=dtype) for _ in range(3)]
    pk, pq = [torch.randn(H, 64, 64, device="cuda", generator=g, dtype=dtype) for _ in range(2)]
    kw = dict(position_buckets=32, max_relative_positions=64, return_lse=True)
    if padded:
        kw["seq_len"] = torch.randint(0, L + 1, (B,), device="cuda", generator=g, dtype=torch.int32)
    (one, one_lse), (shared, shared_lse) = [ops.disentangled_attention_fwd(q, k, v, pk, pq, far_splits=f, near_splits=n, **kw) for f, n in ((1, 1), (far, near))]
    # c2p and the scaled query are rounded alike on both sides; probabilities, against other reference points, partial results and outputs by half an eps each of at most max |v|
    assert (shared - one).abs().max() <= 2.5 * EPS[dtype] * v.abs().max()
    assert (shared_lse - one_lse).nan_to_num(posinf=0, neginf=0).abs().max() <= 1e-5 and torch.equal(shared_lse.isinf(), one_lse.isinf())
