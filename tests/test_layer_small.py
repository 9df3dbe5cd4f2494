"""A layer of short texts in one launch (csrc/fdb_small.hip): against the projections and the attention in 64 bits with the roundings of q, k and v in
between, at the ends of its sizes, with padding on either side, and what is refused."""
import numpy as np
import pytest
import torch

from flashdeberta_amd import _lib, ops
from oracle import disentangled_oracle as O

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
CODE = {torch.bfloat16: _lib.FDB_BF16, torch.float16: _lib.FDB_F16}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("B,L,H,C,buckets,most,bounds", [
    (1, 1, 1, 64, 256, 512, None), (1, 24, 12, 768, 256, 512, None), (2, 31, 3, 128, 256, 512, None), (3, 32, 2, 192, 32, 64, None), (1, 32, 4, 1024, 0, 20, None),
    (1, 33, 2, 64, 256, 512, None), (2, 64, 3, 128, 32, 64, None), (1, 65, 2, 64, 256, 512, None), (1, 97, 2, 128, 32, 64, None), (2, 128, 2, 256, 256, 512, None),
    (1, 128, 3, 320, 16, 16, None), (7, 17, 5, 320, 16, 16, None),   # a table that saturates within the block
    (5, 32, 2, 256, 256, 512, [(0, 32), (0, 1), (3, 29), (31, 1), (10, 0)]), (4, 9, 3, 64, 32, 64, [(-2, 9), (0, 20), (0, -1), (4, 3)]),
    (5, 60, 2, 192, 256, 512, [(0, 60), (0, 32), (0, 33), (27, 33), (5, -1)]), (6, 120, 2, 64, 32, 64, [(0, 120), (0, 64), (0, 65), (119, 1), (20, 33), (0, 97)])])
def test_against_64_bits(B, L, H, C, buckets, most, bounds, dtype):
    g = torch.Generator().manual_seed(B * 100 + L)
    rnd = lambda *s, k=1.0: (torch.randn(*s, generator=g) * k).to(dtype)
    S = ops.att_span(buckets, most)
    x, w, bias, pk, pq = rnd(B, L, C), rnd(3 * H * 64, C + 8, k=C ** -0.5)[:, :C], rnd(3 * H * 64), rnd(2 * S, H, 64), rnd(2 * S + 3, H, 64)
    lut, radius = ops.delta_lut_device(buckets, most, torch.device("cuda", 0))
    starts, lens = zip(*(bounds or [(0, L)] * B))
    d = [t.cuda() for t in (x, pk, pq, bias)]
    wd = rnd(3 * H * 64, C + 8).cuda()   # rows with a stride of their own
    wd[:, :C] = w.cuda()
    out = torch.full((B * L + 1, H * 64), 7.0, dtype=dtype, device="cuda")
    start, length = [torch.tensor(t, dtype=torch.int32, device="cuda") for t in (starts, lens)]
    scale = (3 * 64) ** -0.5
    rc = _lib.lib.fdb_layer_small(d[0].data_ptr(), wd.data_ptr(), d[3].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), out.data_ptr(), start.data_ptr() if bounds else None,
                                  length.data_ptr() if bounds else None, lut.data_ptr(), B, L, H, C, C, C + 8, 64, H * 64, 64, H * 64, S, radius, scale, CODE[dtype],
                                  torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and (out[-1] == 7.0).all()
    got = out[:-1].view(B, L, H, 64).float().cpu().numpy()
    qkv = (x.double() @ w.double().t() + bias.double()).to(dtype).view(B, L, 3, H, 64)   # rounded where the kernel rounds
    n = lambda t: t.float().numpy().astype(np.float64)
    for b in range(B):
        s = min(max(starts[b], 0), L)
        e = s + min(max(lens[b], 0), L - s)
        pad = np.delete(got[b], np.s_[s:e], axis=0)
        assert np.isnan(pad).all() if lens[b] < 0 else (pad == 0).all()
        if s == e:
            continue
        q, k, v = [n(qkv[b:b + 1, s:e, i]).transpose(0, 2, 1, 3) for i in range(3)]
        ref = O.disentangled_attention(q, k, v, n(pk).transpose(1, 0, 2), n(pq).transpose(1, 0, 2)[:, :2 * S], buckets, most)[0].transpose(1, 0, 2)
        # Scores up to about 5 carry a rounding of the scaled query and one of c2p, q, k and v may round the other way at a tie of the sums, the probabilities and
        # the output are rounded: five roundings of values about the size of the result's largest.
        assert np.abs(got[b, s:e] - ref).max() <= 5 * EPS[dtype] * max(1.0, np.abs(ref).max())


def _alone(x, w, bias, pos_key, pos_query, heads, scale, buckets, most, start, length):
    (B, L, C), out = x.shape, torch.empty_like(x)
    lut, radius = ops.delta_lut_device(buckets, most, x.device)
    pk, pq = [t.reshape(heads, -1, 64) if t.dim() == 4 else t for t in (pos_key, pos_query)]
    p = lambda t: None if t is None else t.data_ptr()
    rc = _lib.lib.fdb_layer_small(p(x), p(w), p(bias), p(pk), p(pq), p(out), p(start), p(length), p(lut), B, L, heads, C, C, w.stride(0), pk.stride(0), pk.stride(1), pq.stride(0),
                                  pq.stride(1), ops.att_span(buckets, most), radius, scale, CODE[x.dtype], torch.cuda.current_stream().cuda_stream)
    return rc, out


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,heads,padded", [(1, 24, 12, False), (4, 32, 12, True), (2, 33, 12, True), (21, 20, 12, True), (22, 20, 12, True), (3, 7, 6, False), (2, 64, 12, True), (5, 100, 6, True), (2, 129, 12, True)])
def test_layer_with_and_without(B, L, heads, padded):
    """The module's inference on either side of the sizes it takes, against its projections and the operator one by one, also from a graph."""
    from flashdeberta_amd import DebertaV2Config, FlashDisentangledSelfAttention

    torch.manual_seed(L)
    cfg = DebertaV2Config(hidden_size=64 * heads, num_attention_heads=heads, relative_attention=True, pos_att_type="p2c|c2p", position_buckets=256, max_relative_positions=512,
                          share_att_key=True, attention_probs_dropout_prob=0.0, hidden_dropout_prob=0.0)
    att = FlashDisentangledSelfAttention(cfg).eval().cuda().to(torch.bfloat16)
    x, rel = torch.randn(B, L, 64 * heads, device="cuda").to(torch.bfloat16), torch.randn(512, 64 * heads, device="cuda").to(torch.bfloat16)
    lens = torch.tensor([L] + [max(1, L - 3 * b) for b in range(1, B)], device="cuda")
    mask = (torch.arange(L, device="cuda") < lens[:, None]).long() if padded else None
    with torch.no_grad():
        got = att(x, mask, rel_embeddings=rel)[0]
        # Which way it went: one launch allocates nothing but its result, and has the bits of that launch by itself
        serves = bool(_lib.lib.fdb_layer_small_serves(B, L, heads, 64 * heads))
        allocated = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
        before = allocated()
        again = att(x, mask, rel_embeddings=rel)[0]
        assert (allocated() - before == 1) == serves and torch.equal(got, again)
        if serves:
            rc, alone = _alone(x, *att._native_args(mask, rel, x))
            assert rc == 0 and torch.equal(got, alone)
        handle = att.value_proj.register_forward_hook(lambda *a: None)   # its modules are called
        ref = att(x, mask, rel_embeddings=rel)[0]
        handle.remove()
        assert (got.float() - ref.float()).norm() <= 6e-3 * ref.float().norm()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = att(x, mask, rel_embeddings=rel)[0]
        for k in (1.0, -0.5, 2.0):
            x.mul_(k)
            graph.replay()
            assert torch.equal(captured, att(x, mask, rel_embeddings=rel)[0])


def test_where_it_serves():
    serves = _lib.lib.fdb_layer_small_serves
    assert serves(1, 24, 12, 768) and serves(21, 32, 12, 768) and not serves(22, 32, 12, 768)   # a workgroup a compute unit (256)
    assert not serves(4, 129, 12, 768) and serves(1, 64, 12, 768) and not serves(3, 128, 12, 768) and serves(4, 97, 12, 768) and not serves(1, 24, 12, 100) and not serves(0, 24, 12, 768)


@pytest.mark.parametrize("change,code", [
    (dict(x=0), -1), (dict(w=0), -1), (dict(pk=0), -1), (dict(pq=0), -1), (dict(out=0), -1), (dict(dtype=_lib.FDB_F32), -2), (dict(x=24), -4), (dict(w=40), -4), (dict(bias=52), -4),
    (dict(pk=72), -4), (dict(out=88), -4), (dict(ldx=68), -4), (dict(pqr=68), -4), (dict(batch=0), -5), (dict(seqlen=129), -5), (dict(seqlen=0), -5), (dict(depth=96), -5), (dict(ldw=56), -5),
    (dict(pkr=-64), -5), (dict(pkr=1 << 23), -5), (dict(pkr=1 << 22, span=1 << 9), -5), (dict(span=0), -6), (dict(lut=0), -6), (dict(radius=0), -6)])
def test_refused_on_the_host(change, code):
    kw = dict(x=16, w=32, bias=48, pk=64, pq=80, out=96, start=0, length=0, lut=128, batch=2, seqlen=24, heads=2, depth=64, ldx=64, ldw=64, pkh=64, pkr=64, pqh=64, pqr=64, span=32,
              radius=64, scale=0.1, dtype=_lib.FDB_BF16)
    kw.update(change)
    pointers = ("x", "w", "bias", "pk", "pq", "out", "start", "length", "lut")
    assert _lib.lib.fdb_layer_small(*[v or None if k in pointers else v for k, v in kw.items()], None) == code
