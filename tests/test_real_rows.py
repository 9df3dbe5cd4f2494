"""The projections of a padded batch's real rows (csrc/fdb_gemm.hip): each height of tile, and lengths that put the rows where the look-up can go wrong."""
import random

import pytest
import torch

from flashdeberta_amd import _lib


def _lengths(kind, batch, seqlen):
    rng = random.Random(batch * 1000 + seqlen)
    if kind == "full":
        return [0] * batch, [seqlen] * batch
    if kind == "none":
        return [0] * batch, [0] * batch
    if kind == "one":        # a single real row, in the last sequence; -1: a row nothing is asked of
        return [seqlen - 1] * batch, [-1] * (batch - 1) + [1]
    if kind == "clamped":    # a start and lengths past the sequence
        return [rng.choice([-3, 0, seqlen - 2, seqlen + 5]) for _ in range(batch)], [rng.choice([-1, 0, 1, seqlen, seqlen + 9]) for _ in range(batch)]
    starts = [rng.choice([0, 0, rng.randrange(seqlen)]) for _ in range(batch)]
    return starts, [rng.choice([0, rng.randrange(seqlen + 1 - s), seqlen - s]) if kind == "ragged" else max(1, (seqlen - s) // 3) for s in starts]


@pytest.mark.gpu
@pytest.mark.parametrize("cleared", [False, True], ids=["left", "cleared"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("kind", ["full", "none", "one", "clamped", "ragged", "third"])
@pytest.mark.parametrize("batch,seqlen,N,K", [(1, 1500, 2304, 64), (8, 512, 2304, 128), (64, 33, 1544, 64), (47, 170, 3080, 64), (63, 260, 2304, 64), (5, 2999, 200, 192), (3, 700, 3072, 320)])
def test_real_rows(batch, seqlen, N, K, kind, dtype, cleared):
    g = torch.Generator(device="cuda").manual_seed(batch + N)
    x, w = [(torch.randn(r, K, device="cuda", generator=g) * s).to(dtype) for r, s in ((batch * seqlen, 1.0), (N, K ** -0.5))]
    bias = torch.randn(N, device="cuda", generator=g).to(dtype)
    starts, lens = _lengths(kind, batch, seqlen)
    real = torch.zeros(batch, seqlen, dtype=torch.bool)
    for b in range(batch):
        s = min(max(starts[b], 0), seqlen)
        real[b, s:s + min(max(lens[b], 0), seqlen - s)] = True
    real = real.view(-1).cuda()
    x[~real] = float("nan")   # whatever padding holds
    out = torch.full((batch * seqlen, N), 7.0, device="cuda", dtype=dtype)
    start, length = [torch.tensor(t, dtype=torch.int32, device="cuda") for t in (starts, lens)]
    entry = _lib.lib.fdb_gemm_real_cleared if cleared else _lib.lib.fdb_gemm_real
    assert entry(x.data_ptr(), w.data_ptr(), bias.data_ptr(), out.data_ptr(), None if max(starts) == 0 else start.data_ptr(), length.data_ptr(), batch,
                 seqlen, N, K, K, K, N, {torch.bfloat16: _lib.FDB_BF16, torch.float16: _lib.FDB_F16}[dtype],
                 torch.cuda.current_stream().cuda_stream) == 0
    assert (out[~real] == (0.0 if cleared else 7.0)).all()
    ref = x[real].double() @ w.double().t() + bias.double()
    bound = torch.finfo(dtype).eps / 2 * ref.abs() * 1.01 + 1e-5   # one rounding of the result; the fp32 sums' own is smaller by 2^-10
    assert ((out[real].double() - ref).abs() <= bound).all()


def test_where_it_serves():
    serves = _lib.lib.fdb_gemm_real_serves
    assert serves(8, 512, 2304, 768, 768) and not serves(2, 512, 2304, 768, 768)
    assert not serves(65, 512, 2304, 768, 768) and not serves(8, 512, 2304, 100, 104) and not serves(64, 65536, 2304, 768, 768)


@pytest.mark.parametrize("entry", ["fdb_gemm_real", "fdb_gemm_real_cleared"])
@pytest.mark.parametrize("change,code", [
    (dict(x=0), -1), (dict(w=0), -1), (dict(out=0), -1), (dict(length=0), -1), (dict(dtype=_lib.FDB_F32), -2), (dict(dtype=_lib.FDB_FP8_E4M3), -2),
    (dict(batch=0), -5), (dict(batch=65), -5), (dict(seqlen=0), -5), (dict(batch=64, seqlen=(1 << 18) + 1), -5), (dict(cols=12), -5), (dict(cols=0), -5), (dict(depth=96), -5),
    (dict(depth=32), -5), (dict(ldx=56), -5), (dict(ldw=56), -5), (dict(ldo=56), -5), (dict(ldx=(1 << 22) + 8), -5), (dict(ldw=(1 << 22) + 8), -5),
    (dict(batch=64, seqlen=1 << 18, ldx=64), -5),    # rows of x past 2 GB
    (dict(x=24), -4), (dict(w=40), -4), (dict(out=88), -4), (dict(bias=52), -4), (dict(ldx=68), -4), (dict(ldw=68), -4), (dict(ldo=68), -4)])
def test_refused_on_the_host(change, code, entry):
    kw = dict(x=16, w=32, bias=48, out=80, start=0, length=96, batch=8, seqlen=64, cols=64, depth=64, ldx=64, ldw=64, ldo=64, dtype=_lib.FDB_BF16)
    kw.update(change)
    args = [v or None if k in ("x", "w", "bias", "out", "start", "length") else v for k, v in kw.items()]
    assert getattr(_lib.lib, entry)(*args, None) == code


@pytest.mark.gpu
@pytest.mark.parametrize("side", ["right", "left"])
def test_nothing_reads_the_rows_left_out(side):
    """A layer on a padded batch, forward and backward, where the memory it is given holds zeros and where it holds NaN."""
    from flashdeberta_amd import DebertaV2Config, FlashDisentangledSelfAttention

    torch.manual_seed(0)
    cfg = DebertaV2Config(hidden_size=768, num_attention_heads=12, relative_attention=True, pos_att_type="p2c|c2p", position_buckets=256, max_relative_positions=512,
                          share_att_key=True, attention_probs_dropout_prob=0.0, hidden_dropout_prob=0.0)
    layer = FlashDisentangledSelfAttention(cfg).cuda().to(torch.bfloat16)
    B, L = 9, 500
    x, rel = [torch.randn(*s, 768, device="cuda").to(torch.bfloat16).requires_grad_() for s in ((B, L), (512,))]
    lens = torch.tensor([500, 1, 0, 499, 64, 257, 128, 333, 90], device="cuda")
    at = torch.arange(L, device="cuda")
    mask = ((at < lens[:, None]) if side == "right" else (at >= L - lens[:, None])).long()
    grad = torch.randn(B, L, 768, device="cuda").to(torch.bfloat16)
    seen = []

    def pack(t):   # what a hook on the saved tensors meets: no memory that nobody has written
        assert not t.is_floating_point() or t.isfinite().all(), t.shape
        return t

    for poison in (0.0, float("nan"), float("nan")):
        hold = [torch.full((n,), poison, device="cuda", dtype=torch.bfloat16) for n in [B * L * 2304] * 4 + [B * L * 768] * 6 + [512 * 1536] * 4]
        del hold   # what the calls below are given
        with torch.no_grad():
            inferred = layer.eval()(x, mask, rel_embeddings=rel)[0]
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
            out = layer.train()(x, mask, rel_embeddings=rel)[0]
        seen.append([inferred, out, *torch.autograd.grad(out, [x, rel, *layer.parameters()], grad)])
    assert all(torch.isfinite(t).all() for t in seen[0])
    for other in seen[1:]:
        assert all(torch.equal(a, b) for a, b in zip(seen[0], other))
