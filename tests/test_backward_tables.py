"""The backward with the tables in the kernel (fdb_attn_bwd_tables) and the training node of a layer: against the oracle's chain rule
at the edges of tiles, steps, rings and zones, and against the module-by-module forward under autograd."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from flashdeberta_amd import _lib, ops
from oracle import disentangled_oracle as O


def _np(x):
    return x.detach().float().cpu().numpy().astype(np.float64)


CASES = [
    # B, L, H, buckets, max_rel, causal, (start, length) per row or None
    (1, 1, 1, 256, 512, False, None),
    (2, 32, 2, 256, 512, False, None),
    (1, 33, 1, 256, 512, True, None),
    (1, 129, 3, 32, 64, False, None),                      # one row in the last tile, far steps on both sides
    (2, 160, 2, 32, 64, True, None),
    (1, 544, 1, 256, 512, False, None),                    # the first length with far steps (radius 512)
    (1, 1153, 1, 256, 512, False, None),                   # a tile with far steps on both sides, an odd end
    (1, 900, 2, 256, 512, True, None),
    (3, 300, 2, 32, 64, False, [(0, 300), (37, 200), (299, 1)]),   # left and right padding, a row of one token
    (2, 257, 1, 16, 16, False, [(0, 0), (1, 256)]),        # an empty row; a table that saturates within a step
    (1, 300, 1, 256, 200, False, None),                    # steps of several table rows per position
    (1, 400, 2, 0, 100, False, None),                      # no buckets
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%dL%dH%d_b%d_m%d_c%d%s" % (c[:6] + ("pad" if c[6] else "",)))
def test_table_backward_matches_oracle(case, dtype):
    B, L, H, pb, mr, causal, rows = case
    S, D = ops.att_span(pb, mr), 64
    g = torch.Generator().manual_seed(L * 7 + H)
    q, k, v, dout = [torch.randn(B, L, H, D, generator=g).to(dtype) for _ in range(4)]
    pk, pq = [torch.randn(H, 2 * S, D, generator=g).to(dtype) for _ in range(2)]
    kw = dict(position_buckets=pb, max_relative_positions=mr, causal=causal)
    if rows:
        kw["seq_start"], kw["seq_len"] = [torch.tensor(x, dtype=torch.int32).cuda() for x in zip(*rows)]
    c = [x.cuda() for x in (q, k, v, pk, pq)]
    out, lse = ops.disentangled_attention_fwd(*c, return_lse=True, **kw)
    got = ops.disentangled_attention_bwd(*c[:3], out, lse, dout.cuda(), *c[3:], **kw)
    again = ops.disentangled_attention_bwd(*c[:3], out, lse, dout.cuda(), *c[3:], **kw)
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    ref = [np.zeros((B, L, H, D)) for _ in range(3)] + [np.zeros((H, 2 * S, D)) for _ in range(2)]
    t = lambda x, b, s: _np(x[b:b + 1, s]).transpose(0, 2, 1, 3)
    for b, (start, length) in enumerate(rows or [(0, L)] * B):
        if not length:
            continue
        s = slice(start, start + length)
        r = O.disentangled_attention_backward(*[t(x, b, s) for x in (q, k, v, dout)], _np(pk), _np(pq), pb, mr, causal=causal)
        for n in range(3):
            ref[n][b:b + 1, s] = r[n].transpose(0, 2, 1, 3)
        ref[3] += r[3]
        ref[4] += r[4]
    _check(got, ref, dtype)


def _check(got, ref, dtype):
    """Scores, probabilities or score gradients, and results are rounded to the type once each, to half its epsilon at most and independently
    of one another: together less than the epsilon in the 2-norm of a gradient (measured: 0.2 to 0.5).  A single entry may owe its error to
    a few large terms: three epsilons of the largest entry (measured: 0.3 to 1.4).  Gradients that cancel to nothing have the floor."""
    eps = torch.finfo(dtype).eps
    for name, a, r in zip(("dq", "dk", "dv", "dK_r", "dQ_r"), got, ref):
        off = np.abs(_np(a) - r)
        assert np.isfinite(off).all(), name
        assert np.linalg.norm(off) <= eps * max(np.linalg.norm(r), 1e-2 * r.size ** 0.5), "%s: %.2f epsilons" % (name, np.linalg.norm(off) / np.linalg.norm(r) / eps)
        assert off.max() <= 3 * eps * max(np.abs(r).max(), 1e-2), "%s: err %.3e, largest %.3e" % (name, off.max(), np.abs(r).max())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_saturated_rows_of_a_key_that_all_queries_attend_to(dtype):
    """Loss-scaled gradients: the far queries' score gradients of one key add up to 1.4e5, beyond fp16, while everything that leaves
    the backward (which takes the soft-max scale, 1 / 13.9) is finite there."""
    B, L, H, D, pb, mr = 1, 900, 1, 64, 32, 64
    g = torch.Generator().manual_seed(3)
    q = 1.2 + 0.05 * torch.randn(B, L, H, D, generator=g)
    k, v = [0.05 * torch.randn(B, L, H, D, generator=g) for _ in range(2)]
    k[:, 0] += 1.2          # q . k_0 / 13.9 = 6.6: half of every row's probability
    v[:, 0] += 12.0         # dO . v_0 = 770
    dout = 1.0 + 0.05 * torch.randn(B, L, H, D, generator=g)
    pk, pq = [0.05 * torch.randn(H, 2 * pb, D, generator=g) for _ in range(2)]
    q, k, v, dout, pk, pq = [x.to(dtype) for x in (q, k, v, dout, pk, pq)]
    kw = dict(position_buckets=pb, max_relative_positions=mr)
    c = [x.cuda() for x in (q, k, v, pk, pq)]
    out, lse = ops.disentangled_attention_fwd(*c, return_lse=True, **kw)
    got = ops.disentangled_attention_bwd(*c[:3], out, lse, dout.cuda(), *c[3:], **kw)
    t = lambda x: _np(x).transpose(0, 2, 1, 3)
    ref = O.disentangled_attention_backward(*[t(x) for x in (q, k, v, dout)], _np(pk), _np(pq), pb, mr)
    ref = [r.transpose(0, 2, 1, 3) for r in ref[:3]] + list(ref[3:])
    # the sum itself, from what it becomes: d pos_query of the saturated rows is the far sums of all keys times the keys
    assert np.abs(ref[4]).max() * np.sqrt(3 * D) / 1.3 > 65504 > max(np.abs(r).max() for r in ref)
    _check(got, ref, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("B,L", [(2, 96), (1, 700)])
def test_gradient_of_any_layout(B, L):
    """The gradient of the output as autograd hands it over -- expanded (the output's sum), transposed, rows with a stride of their own, no
    unit stride, reversed roles of batch and heads -- gives the bits of its contiguous copy."""
    H, D = 3, 64
    g = torch.Generator(device="cuda").manual_seed(L)
    normal = lambda *s: torch.randn(*s, device="cuda", generator=g).to(torch.float16)
    leaves = [normal(B, H, L, D).requires_grad_() for _ in range(3)] + [normal(H, 64, D).requires_grad_() for _ in range(2)]
    out = ops.flash_attention_with_disentangled(*leaves, position_buckets=32, max_relative_distance=64)
    forms = [normal(1, 1, 1, 1).expand(B, H, L, D), normal(1, 1, 1, D).expand(B, H, L, D), normal(B, L, H, D).transpose(1, 2),
             normal(B, H, L, D + 16)[..., 8:D + 8], normal(B, H, D, L).transpose(2, 3), normal(H, B, L, D).transpose(0, 1), normal(B, H, 1, D).expand(B, H, L, D)]
    for dout in forms:
        got = torch.autograd.grad(out, leaves, dout, retain_graph=True)
        ref = torch.autograd.grad(out, leaves, dout.contiguous(), retain_graph=True)
        assert all(torch.equal(a, b) for a, b in zip(got, ref)), dout.stride()
    total = torch.autograd.grad(out.sum(), leaves, retain_graph=True)
    ref = torch.autograd.grad(out, leaves, torch.ones_like(out))
    assert all(torch.equal(a, b) for a, b in zip(total, ref))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,rows2,cols2", [(1, 8, 0, 0), (63, 512, 5, 8), (64, 520, 64, 512), (3, 16, 200, 8), (65, 2304, 512, 1536), (4096, 768, 0, 0)])
def test_column_sums(rows, cols, rows2, cols2):
    x = torch.randn(rows, cols, device="cuda").to(torch.bfloat16)
    y = torch.randn(rows2, cols2, device="cuda").to(torch.bfloat16) if rows2 else None
    out = torch.empty(cols, device="cuda", dtype=torch.bfloat16)
    ws = torch.empty(_lib.lib.fdb_column_sums_workspace_bytes(rows, cols, rows2), dtype=torch.uint8, device="cuda")
    assert _lib.lib.fdb_column_sums(x.data_ptr(), rows, cols, None if y is None else y.data_ptr(), rows2, cols2, out.data_ptr(), ws.data_ptr(), 1,
                                    torch.cuda.current_stream().cuda_stream) == 0
    ref = x.float().sum(0)
    if y is not None:
        ref[:cols2] += y.float().sum(0)
    assert ((out.float() - ref).abs() <= 4e-3 * ref.abs() + 1e-4 * rows ** 0.5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,padded,dropout", [(1, 7, False, 0.0), (3, 200, True, 0.0), (2, 640, False, 0.0), (3, 200, True, 0.25)])
def test_layer_node_matches_separate_projections(B, L, padded, dropout):
    """The whole layer as one node against the same module with its projections called one by one (a hook on one of them
    turns the node off): output and every gradient, with the same relative embeddings dropped on either side."""
    from flashdeberta_amd import DebertaV2Config, FlashDisentangledSelfAttention

    torch.manual_seed(L)
    cfg = DebertaV2Config(hidden_size=192, num_attention_heads=3, relative_attention=True, pos_att_type="p2c|c2p", position_buckets=32,
                          max_relative_positions=64, share_att_key=True, hidden_dropout_prob=dropout, attention_probs_dropout_prob=0.0)
    att = FlashDisentangledSelfAttention(cfg).train().cuda().to(torch.bfloat16)
    x = torch.randn(B, L, 192, device="cuda").to(torch.bfloat16).requires_grad_()
    rel = torch.randn(64, 192, device="cuda").to(torch.bfloat16).requires_grad_()
    mask = torch.ones(B, L, device="cuda", dtype=torch.long)
    if padded:
        mask[0, L // 3:] = 0
    dout = torch.randn(B, L, 192, device="cuda").to(torch.bfloat16)
    leaves = [x, rel, *att.parameters()]

    def grads():
        torch.manual_seed(99)   # of the dropout
        out = att(x, mask, rel_embeddings=rel)[0]
        return (out.detach(), out.grad_fn.name(), *torch.autograd.grad(out, leaves, dout))

    one = grads()
    handle = att.value_proj.register_forward_hook(lambda *a: None)
    separate = grads()
    handle.remove()
    assert one[1] != separate[1]
    if dropout:
        # the gradient of the relative embeddings; module by module it is a sum of two rounded ones, which may cancel exactly, too
        dropped = one[3] == 0
        assert 0.2 < dropped.float().mean() < 0.3 and not separate[3][dropped].any()
    for a, b in zip(one[:1] + one[2:], separate[:1] + separate[2:]):
        assert (a.float() - b.float()).norm() <= 2e-2 * b.float().norm()
    # only what is asked for
    att.value_proj.weight.requires_grad_(False)
    torch.manual_seed(99)
    some = torch.autograd.grad(att(x, mask, rel_embeddings=rel)[0], [x, att.query_proj.bias], dout)
    assert torch.equal(some[0], one[2]) and some[1].shape == (192,)


@pytest.mark.gpu
def test_node_replays_from_a_graph_and_through_saved_tensor_hooks():
    """Forward and backward of the operator in a captured graph, replayed with eager work between, and with the saved tensors taken to
    the host and back: the eager call's bits."""
    B, H, L, D = 1, 2, 700, 64
    leaves = [torch.randn(*s, device="cuda").to(torch.bfloat16).requires_grad_() for s in ((B, H, L, D),) * 3 + ((H, 512, D),) * 2]
    dout = torch.randn(B, H, L, D, device="cuda").to(torch.bfloat16)

    def step():
        out = ops.flash_attention_with_disentangled(*leaves, position_buckets=256, max_relative_distance=512)
        return (out.detach(), *torch.autograd.grad(out, leaves, dout))

    ref = step()
    with torch.autograd.graph.save_on_cpu():
        assert all(torch.equal(a, b) for a, b in zip(step(), ref))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for scale in (1.0, 0.5, 2.0):
        with torch.no_grad():
            leaves[0].mul_(scale)
        ref = step()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(captured, ref))


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,H,rows", [
    (1, 1100, 26, None),                                   # one share of more row blocks than the tables of what is there hold (32 turns)
    (1, 2300, 12, None),                                   # several such shares, the last of them shorter
    (2, 2300, 12, [(9, 2222), (0, 71)]),                   # shares of equal numbers of row blocks
    (7, 700, 12, [(0, 700), (0, 0), (699, 1), (0, 33), (100, 600), (0, 320), (37, 511)]),   # shares that begin and end inside sequences
    (64, 130, 6, [(n % 5, 2 * n) for n in range(64)]),
])
def test_table_gradients_of_any_share(B, L, H, rows):
    """The tables' gradients of all heads in one call, few and large shares of the tokens, against one call a head, many and small ones: both round the same
    sums to the type once, so they differ by its epsilon at most, and by the order of the fp32 sums."""
    dtype = torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(L + H)
    q, k, v, dout = [torch.randn(B, L, H, 64, device="cuda", generator=g).to(dtype) for _ in range(4)]
    pk, pq = [torch.randn(H, 512, 64, device="cuda", generator=g).to(dtype) for _ in range(2)]
    kw = dict(position_buckets=256, max_relative_positions=512)
    if rows:
        kw["seq_start"], kw["seq_len"] = [torch.tensor(x, dtype=torch.int32).cuda() for x in zip(*rows)]
    out, lse = ops.disentangled_attention_fwd(q, k, v, pk, pq, return_lse=True, **kw)
    got = ops.disentangled_attention_bwd(q, k, v, out, lse, dout, pk, pq, **kw)[3:]
    ref = [torch.zeros_like(pk), torch.zeros_like(pq)]
    for h in range(H):
        one = [x[:, :, h:h + 1].contiguous() for x in (q, k, v, out)] + [lse[:, h:h + 1].contiguous(), dout[:, :, h:h + 1].contiguous()]
        for r, x in zip(ref, ops.disentangled_attention_bwd(*one, pk[h:h + 1], pq[h:h + 1], **kw)[3:]):
            r[h:h + 1] = x
    eps = torch.finfo(dtype).eps
    for a, r in zip(got, ref):
        a, r = a.double(), r.double()
        off = (a - r).abs() - eps * r.abs()
        assert float(off.max()) <= 2.0 ** -24 * L * float(r.abs().max()), "%.3e of %.3e" % (float(off.max()), float(r.abs().max()))
