"""The native host path (csrc/fdb_torch.cpp) and the linear kernels (csrc/fdb_linear.hip): mask bounds against
padding.seq_bounds, products against fp32 torch, the one-call encoder layer against the module-by-module one."""
import sys
import threading
from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F

from flashdeberta_amd import _lib, model
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


def _rel(a, b):
    return ((a.float() - b).norm() / b.norm()).item()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,code,tol", [(torch.bfloat16, 1, 4e-3), (torch.float16, 2, 6e-4)], ids=["bf16", "fp16"])
@pytest.mark.parametrize("M,N,K", [
    (1, 2, 32), (16, 48, 64), (17, 768, 768), (32, 18, 96), (24, 768, 3072),   # weights streamed, eight and sixteen waves
    (33, 64, 64), (64, 100, 128), (65, 132, 192), (257, 768, 768),              # tiles: one step, odd counts, ragged edges
    (40, 18, 96), (70, 30, 64),                                                 # many rows, sizes the tiles do not take
])
def test_linear_kernels(M, N, K, dtype, code, tol):
    g = torch.Generator(device="cuda").manual_seed(M * N + K)
    x, w = [torch.randn(r, K + 8, device="cuda", generator=g).to(dtype)[:, :K] for r in (M, N)]   # rows with a stride of their own
    b = torch.randn(N, device="cuda", generator=g).to(dtype)
    out = torch.full((M + 1, N), 7.0, device="cuda", dtype=dtype)
    for bias in (b, None):
        rc = _lib.lib.fdb_linear(x.data_ptr(), w.data_ptr(), None if bias is None else bias.data_ptr(), out.data_ptr(), M, N, K, x.stride(0),
                                 w.stride(0), N, code, torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        ref = F.linear(x.float(), w.float(), None if bias is None else bias.float())
        assert _rel(out[:M], ref) < tol and (out[M] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("M,N,K", [(1, 768, 768), (24, 2304, 768), (301, 768, 3072), (4096, 3072, 768)])
def test_library_products_have_the_bits_of_torch(M, N, K, dtype):
    x, w, b = [torch.randn(*s, device="cuda").to(dtype) for s in ((M, K), (N, K), (N,))]
    assert torch.equal(_lib.native.linear(x, w, b, False), F.linear(x, w, b))


# Every form of a product that a layer has: (transposed a, transposed b, bias, accumulated, a with 2 dimensions, 3, or 3
# with one of them of size one and any stride); the rows that take part are the first of more.
FORMS = [(False, True, True, False, 3), (False, True, True, False, 4), (False, True, True, False, 2), (False, False, False, False, 2), (True, False, False, False, 3),
         (True, False, False, True, 2)]


@pytest.mark.parametrize("route", [pytest.param(("cpu", False), id="torch_cpu"), pytest.param(("cuda", False), id="torch", marks=pytest.mark.gpu),
                                   pytest.param(("cuda", True), id="library", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("form", FORMS, ids=lambda f: "%s%s%s%s%d" % ("t" if f[0] else "n", "t" if f[1] else "n", "b" if f[2] else "", "+" if f[3] else "", f[4]))
def test_products_and_their_second_route(form, route):
    """hipBLASLt's product and the one that stands in where it has no kernel compute the same forms."""
    trans_a, trans_b, with_bias, accumulate, dims = form
    device, library = route
    m, n, k = 48, 32, 64
    g = torch.Generator().manual_seed(m + sum(form))
    normal = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(device)
    rows_a, rows_b = (k, n if trans_b else k) if trans_a else (m, n if trans_b else k)
    cols_a = m if trans_a else k
    a = normal(rows_a + 16, cols_a) if dims == 2 else normal(2, rows_a // 2, cols_a) if dims == 3 else normal(2, rows_a, cols_a)[1:].transpose(0, 1)
    assert dims == 2 or a.is_contiguous()
    b, d, bias = normal(rows_b + 16, k if trans_b else n), normal(m + 16, n), normal(n + 16) if with_bias else None
    before = d.clone()
    assert _lib.native.product(a, rows_a, trans_a, b, rows_b, trans_b, d, m, bias, accumulate, library) is True
    x, y = a.reshape(-1, a.shape[-1])[:rows_a].double(), b[:rows_b].double()
    ref = (x.t() if trans_a else x) @ (y.t() if trans_b else y)
    if with_bias:
        ref = ref + bias[:n].double()
    if accumulate:
        ref = ref + before[:m].double()
    assert torch.equal(d[m:], before[m:])
    assert ((d[:m].double() - ref).norm() / ref.norm()).item() <= 2.0 ** -8   # one rounding of the result to bf16


@pytest.mark.gpu
@pytest.mark.parametrize("B,L", [(1, 5), (2, 40), (3, 300), (6, 384)])   # each way of computing the projections
def test_encoder_layer_matches_the_module_by_module_forward(B, L):
    from transformers.models.deberta_v2.modeling_deberta_v2 import DebertaV2Layer

    from flashdeberta_amd import DebertaV2Config, FlashDebertaV2Model

    torch.manual_seed(L)
    cfg = DebertaV2Config(vocab_size=100, hidden_size=256, num_hidden_layers=1, num_attention_heads=4, intermediate_size=1024,
                          relative_attention=True, pos_att_type="p2c|c2p", position_buckets=32, max_relative_positions=64, share_att_key=True,
                          norm_rel_ebd="layer_norm", position_biased_input=False, initializer_range=0.2)
    model = FlashDebertaV2Model(cfg).eval().cuda().to(torch.bfloat16)
    layer = model.encoder.layer[0]
    x = torch.randn(B, L, 256, device="cuda").to(torch.bfloat16)
    mask = torch.ones(B, L, device="cuda", dtype=torch.long)
    mask[-1, L // 2:] = 0
    rel = torch.randn(64, 256, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        got = layer(x, mask, rel_embeddings=rel)[0]
        ref = DebertaV2Layer.forward(layer, x, mask, rel_embeddings=rel)[0]
        assert torch.equal(got, ref)
        calls = []
        handle = layer.output.dense.register_forward_hook(lambda *a: calls.append(1))   # a hook on any part is honoured
        layer(x, mask, rel_embeddings=rel)
        handle.remove()
        assert calls


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("width", [768, 1024])
@pytest.mark.parametrize("B,L", [(2, 40), (3, 300), (6, 256), (8, 384), (5, 999)])   # every tile, and from (8, 384) on the products of real rows
def test_encoder_layer_bits_at_the_widths_of_the_models(B, L, width, dtype):
    """The layer as one call against its modules, and its attention against the library's product of all rows."""
    from transformers.models.deberta_v2.modeling_deberta_v2 import DebertaV2Layer

    from flashdeberta_amd import DebertaV2Config, FlashDebertaV2Model, ops

    torch.manual_seed(width + L)
    cfg = DebertaV2Config(vocab_size=100, hidden_size=width, num_hidden_layers=1, num_attention_heads=width // 64, intermediate_size=4 * width,
                          relative_attention=True, pos_att_type="p2c|c2p", position_buckets=32, max_relative_positions=64, share_att_key=True,
                          norm_rel_ebd="layer_norm", position_biased_input=False, initializer_range=0.05)
    layer = FlashDebertaV2Model(cfg).eval().cuda().to(dtype).encoder.layer[0]
    x, rel = torch.randn(B, L, width, device="cuda").to(dtype), torch.randn(64, width, device="cuda").to(dtype)
    lengths = torch.tensor([L] + [L - (b * L) // (B + 1) for b in range(1, B)], device="cuda")
    mask = (torch.arange(L, device="cuda") < lengths[:, None]).long()
    with torch.no_grad():
        assert torch.equal(layer(x, mask, rel_embeddings=rel)[0], DebertaV2Layer.forward(layer, x, mask, rel_embeddings=rel)[0])
        att = layer.attention.self
        q, k, v = [F.linear(x, p.weight, p.bias).view(B, L, -1, 64) for p in (att.query_proj, att.key_proj, att.value_proj)]
        pk, pq = [F.linear(rel, p.weight, p.bias).view(64, -1, 64).transpose(0, 1) for p in (att.key_proj, att.query_proj)]
        ref = ops.disentangled_attention_fwd(q, k, v, pk, pq, position_buckets=32, max_relative_positions=64, seq_len=lengths.int())
        assert torch.equal(att(x, mask, rel_embeddings=rel)[0], ref.view(B, L, width))


def _encoder_layer(dropout=0.1):
    from flashdeberta_amd import DebertaV2Config, FlashDebertaV2Model

    cfg = DebertaV2Config(vocab_size=100, hidden_size=128, num_hidden_layers=1, num_attention_heads=2, intermediate_size=256, relative_attention=True,
                          pos_att_type="p2c|c2p", position_buckets=32, max_relative_positions=64, share_att_key=True, norm_rel_ebd="layer_norm",
                          position_biased_input=False, hidden_dropout_prob=dropout)
    return FlashDebertaV2Model(cfg).eval().to(torch.bfloat16).encoder.layer[0]


def _takes_one_call(layer):
    """Whether the layer's inference on GPU activations would be the one native call (the decision itself needs no GPU)."""
    hidden = SimpleNamespace(dtype=torch.bfloat16, is_cuda=True, shape=torch.Size((1, 8, 128)))
    with torch.no_grad():
        return layer._native_args(hidden, None, torch.zeros(64, 128, dtype=torch.bfloat16)) is not None


@pytest.mark.parametrize("name", ["attention.output", "output"])
def test_one_call_layer_leaves_no_dropout_out(name):
    """Dropout kept on in an eval model, with a hook, or replaced by another module: transformers' own forward calls it."""
    assert _takes_one_call(_encoder_layer())
    layer = _encoder_layer()
    part = layer.get_submodule(name)
    part.dropout.train()
    assert not _takes_one_call(layer)
    part.dropout.p = 0.0   # on, and dropping nothing
    assert _takes_one_call(layer)
    for register in ("register_forward_hook", "register_forward_pre_hook"):
        handle = getattr(part.dropout, register)(lambda *a: None)
        assert not _takes_one_call(layer)
        handle.remove()
    part.dropout = torch.nn.Linear(128, 128)
    assert not _takes_one_call(layer)


def _changes(part):
    """Ways in which a program changes what calling a module does, each with its undoing."""
    handles = [part.register_forward_hook, part.register_forward_pre_hook, part.register_full_backward_hook]
    for register in handles:
        handle = register(lambda *a: None)
        yield
        handle.remove()
    part.forward = part.forward
    yield
    del part.forward
    cls, old = type(part), type(part).forward
    cls.forward = lambda self, *a, **k: old(self, *a, **k)
    try:
        yield
    finally:
        cls.forward = old
    part.__class__ = type("Other", (cls,), {})
    yield
    part.__class__ = cls


PARTS = ["attention", "attention.self", "attention.self.query_proj", "attention.self.key_proj", "attention.self.value_proj", "attention.output",
         "attention.output.dense", "attention.output.dropout", "attention.output.LayerNorm", "intermediate", "intermediate.dense",
         "intermediate.intermediate_act_fn", "output", "output.dense", "output.dropout", "output.LayerNorm"]


@pytest.mark.parametrize("name", PARTS)
def test_one_call_layer_leaves_changed_parts_to_their_own_call(name):
    layer = _encoder_layer()
    for _ in _changes(layer.get_submodule(name)):
        assert not _takes_one_call(layer)
    assert _takes_one_call(layer)


@pytest.mark.parametrize("name", ["query_proj", "key_proj", "value_proj"])
def test_changed_projections_are_called(name):
    """The attention's own ways round its projections' calls: the concatenated weights, the remembered tables, the training node."""
    att = _attention("cpu")
    rel = torch.randn(64, 128).to(torch.bfloat16)
    called = []
    plain = torch.nn.Linear.forward

    def fused(att):
        with torch.no_grad():
            return att.eval()._native_args(None, rel) is not None, att.train()._trains_as_one_node()

    assert fused(att) == (True, True)
    for _ in _changes(att.get_submodule(name)):
        assert fused(att) == (False, False)
    part = att.get_submodule(name)
    part.forward = lambda x: called.append(1) or plain(part, x)
    with torch.no_grad():
        att.eval()._qkv(rel[None], rel[None])
        assert len(called) == 1
        att._pos_layers(rel)
        att._pos_layers(rel)
    assert len(called) == (1 if name == "value_proj" else 3)   # the tables are not remembered past a forward nobody has looked into
    del part.forward
    assert fused(att) == (True, True)


@pytest.mark.parametrize("how", ["on", "hook", "forward"])
@pytest.mark.parametrize("node", [True, False], ids=["node", "no_node"])
def test_dropout_of_the_relative_embeddings_is_called_once(node, how, monkeypatch):
    """In an eval module, whether anything is recorded or not, and whether or not the training node takes the call."""
    att = _attention("cpu", hidden_dropout_prob=0.5).eval()
    rel, x = torch.randn(64, 128).to(torch.bfloat16), torch.randn(1, 8, 128).to(torch.bfloat16)
    calls, seen = [], []
    if how == "forward":
        att.pos_dropout.forward = lambda r: calls.append(1) or r * 2
    else:
        att.pos_dropout.train(how == "on")
        att.pos_dropout.register_forward_hook(lambda *a: calls.append(1)) if how == "hook" else None

    def layer_node(hidden, rel, *rest):
        seen.append(rel)
        return hidden if node else None

    monkeypatch.setattr(model, "native", SimpleNamespace(layer_node=layer_node, untouched=_lib.native.untouched))
    monkeypatch.setattr(model.ops, "disentangled_attention", lambda q, k, v, pos_key, pos_query, **kw: seen.append(pos_key) or q)
    att(x, None, rel_embeddings=rel)   # recorded: the weights require gradients
    assert len(seen) == (1 if node else 2)
    given = seen[0].detach()
    if how == "on":
        assert (given == 0).any() and ((given == 0) | (given == (2 * rel).to(given.dtype))).all()
    else:
        assert torch.equal(given, rel * 2 if how == "forward" else rel) and len(calls) == 1
    if not node:
        assert torch.equal(seen[1], F.linear(given, att.key_proj.weight, att.key_proj.bias).view(64, 2, 64).transpose(0, 1))
    with torch.no_grad():   # not recorded: the tables are not remembered past a dropout that is more than nothing
        att._pos_layers(rel)
        first, second = att._pos_layers(rel)[0], att._pos_layers(rel)[0]
    assert not torch.equal(first, second) if how == "on" else len(calls) == 4


def _replica(module):
    """What DataParallel computes on each device: a module whose weights are attributes carrying the graph back to the parameters."""
    copy = module._replicate_for_data_parallel()
    for name, child in module._modules.items():
        copy._modules[name] = _replica(child)
    for name, p in module._parameters.items():
        setattr(copy, name, p * 1) if p is not None else copy._parameters.__setitem__(name, None)
    return copy


@pytest.mark.parametrize("share", [True, False], ids=["shared", "separate"])
def test_weights_that_are_no_parameters_are_recorded(share):
    """Eval mode with gradients on: a replica's projections, and any single weight that is not frozen, keep the inference paths off."""
    att = _attention("cpu", share_att_key=share).eval()
    rel, x = torch.randn(64, 128).to(torch.bfloat16), torch.randn(1, 8, 128).to(torch.bfloat16)

    def recorded(a):
        q, k, v = a._qkv(x, x)
        pos_key, pos_query = a._pos_layers(rel)
        return a._native_args(None, rel, x) is None, [t.requires_grad for t in (q, k, v, pos_key, pos_query)]

    replica = _replica(att)
    assert not list(replica.parameters())
    assert recorded(replica) == (True, [True] * 5)
    replica._qkv(x, x)[2].float().sum().backward()
    assert att.value_proj.weight.grad is not None
    for p in att.parameters():
        p.requires_grad_(False)
    assert recorded(att) == (False, [False] * 5)
    for name, expected in (("query_proj", [1, 0, 0, 0, share]), ("key_proj", [0, 1, 0, share, 0]), ("value_proj", [0, 0, 1, 0, 0])) + \
            (() if share else (("pos_key_proj", [0, 0, 0, 1, 0]), ("pos_query_proj", [0, 0, 0, 0, 1]))):
        p = att.get_submodule(name).weight.requires_grad_(True)
        assert recorded(att) == (True, [bool(e) for e in expected]), name
        p.requires_grad_(False)


@pytest.mark.parametrize("norm", ["layer_norm", "none"])
def test_relative_embeddings_of_a_recorded_forward_carry_their_graph(norm):
    """Fine-tuning an eval model: what the encoder hands to its layers leads back to the table and its norm, also of a replica."""
    from flashdeberta_amd import DebertaV2Config, FlashDebertaV2Model

    cfg = DebertaV2Config(vocab_size=100, hidden_size=128, num_hidden_layers=1, num_attention_heads=2, intermediate_size=256, relative_attention=True,
                          pos_att_type="p2c|c2p", position_buckets=32, max_relative_positions=64, share_att_key=True, norm_rel_ebd=norm)
    encoder = FlashDebertaV2Model(cfg).eval().encoder
    seen = []

    class Layer(torch.nn.Module):
        def forward(self, hidden_states, attention_mask, rel_embeddings=None, **kwargs):
            seen.append(rel_embeddings)
            return hidden_states, None

    encoder.layer = torch.nn.ModuleList([Layer()])
    x, mask = torch.randn(1, 8, 128), torch.ones(1, 8)
    run = lambda e: e(x, mask) and seen.pop()
    leaves = [encoder.rel_embeddings.weight] + ([encoder.LayerNorm.weight, encoder.LayerNorm.bias] if norm == "layer_norm" else [])
    for _ in range(2):
        assert all(g is not None for g in torch.autograd.grad(run(encoder).sum(), leaves, allow_unused=True))
    assert all(g is not None for g in torch.autograd.grad(run(_replica(encoder)).sum(), leaves, allow_unused=True))
    with torch.no_grad():
        assert run(encoder) is run(encoder)
    for p in leaves:
        p.requires_grad_(False)
    assert run(encoder) is run(encoder) and not run(encoder).requires_grad
    if norm == "layer_norm":
        for _ in _changes(encoder.LayerNorm):
            assert run(encoder) is not run(encoder)


@pytest.mark.gpu
def test_gradients_of_an_eval_model_are_those_of_training_without_dropout():
    from flashdeberta_amd import DebertaV2Config, FlashDebertaV2Model

    torch.manual_seed(13)
    cfg = DebertaV2Config(vocab_size=100, hidden_size=128, num_hidden_layers=2, num_attention_heads=2, intermediate_size=256, relative_attention=True,
                          pos_att_type="p2c|c2p", position_buckets=32, max_relative_positions=64, share_att_key=True, norm_rel_ebd="layer_norm",
                          position_biased_input=False, hidden_dropout_prob=0.0, attention_probs_dropout_prob=0.0)
    net = FlashDebertaV2Model(cfg).cuda().to(torch.bfloat16)
    ids, mask = torch.randint(0, 100, (2, 60), device="cuda"), torch.ones(2, 60, device="cuda", dtype=torch.long)
    mask[1, 40:] = 0
    names, leaves = zip(*[(n, p) for n, p in net.named_parameters() if p.requires_grad])
    got = []
    for mode in (True, False, False):
        out = net.train(mode)(input_ids=ids, attention_mask=mask).last_hidden_state
        got.append(torch.autograd.grad((out * mask[:, :, None]).float().square().sum(), leaves, allow_unused=True))
    for name, a, *rest in zip(names, *got):
        assert all(torch.equal(a, b) if a is not None else b is None for b in rest), name
        assert a is not None or "rel_embeddings" not in name


@pytest.mark.gpu
def test_dropout_kept_on_in_an_eval_model():
    layer = _encoder_layer(0.5).cuda()
    x, rel = torch.randn(2, 40, 128, device="cuda").to(torch.bfloat16), torch.randn(64, 128, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        first = layer(x, None, rel_embeddings=rel)[0]
        assert torch.equal(first, layer(x, None, rel_embeddings=rel)[0])
        layer.output.dropout.train()
        sampled = [layer(x, None, rel_embeddings=rel)[0] for _ in range(2)]
    assert not torch.equal(*sampled)


def _attention(device="cuda", hidden_dropout_prob=0.0, share_att_key=True, **kw):
    from flashdeberta_amd import DebertaV2Config, FlashDisentangledSelfAttention

    torch.manual_seed(5)
    cfg = DebertaV2Config(hidden_size=128, num_attention_heads=2, relative_attention=True, pos_att_type="p2c|c2p", position_buckets=32,
                          max_relative_positions=64, share_att_key=share_att_key, hidden_dropout_prob=hidden_dropout_prob,
                          attention_probs_dropout_prob=0.0, **kw)
    return FlashDisentangledSelfAttention(cfg).to(device).to(torch.bfloat16)


@pytest.mark.gpu
def test_remembered_values_stay_on_their_stream():
    att = _attention().eval()
    rel, mask = torch.randn(64, 128, device="cuda").to(torch.bfloat16), torch.ones(2, 40, device="cuda")
    remembered = lambda: (att._fused_qkv()[0], att._pos_layers(rel)[0], att._bounds(mask)[1])
    same = lambda a, b: [x is y for x, y in zip(a, b)] == [True] * 3
    streams = [torch.cuda.current_stream()] + [torch.cuda.Stream() for _ in range(6)]
    torch.cuda.synchronize()
    with torch.no_grad():
        seen = []
        for stream in streams[:4]:
            with torch.cuda.stream(stream):
                seen.append(remembered())
                assert same(remembered(), seen[-1])
        assert all(not any(x is y for x, y in zip(a, b)) for i, a in enumerate(seen) for b in seen[:i])
        for stream, values in zip(streams, seen):   # taking turns, each stream finds its own
            with torch.cuda.stream(stream):
                assert same(remembered(), values)
        for stream in streams[4:]:   # no more than a few are kept
            with torch.cuda.stream(stream):
                remembered()
        assert not any(x is y for x, y in zip(remembered(), seen[0]))
        torch.cuda.synchronize()


@pytest.mark.gpu
def test_captured_encoder_follows_its_mask_and_weights():
    """A graph recorded after eager calls on the same mask and weights: replays see what has been written into either since, and eager
    calls between them do not take what only a replay computes."""
    from flashdeberta_amd import DebertaV2Config, FlashDebertaV2Model

    torch.manual_seed(11)
    cfg = DebertaV2Config(vocab_size=100, hidden_size=128, num_hidden_layers=2, num_attention_heads=2, intermediate_size=256, relative_attention=True,
                          pos_att_type="p2c|c2p", position_buckets=32, max_relative_positions=64, share_att_key=True, norm_rel_ebd="layer_norm",
                          position_biased_input=False, initializer_range=0.2)
    net = FlashDebertaV2Model(cfg).eval().cuda().to(torch.bfloat16)
    ids = torch.randint(0, 100, (3, 50), device="cuda")
    lengths = lambda *n: (torch.arange(50, device="cuda") < torch.tensor(n, device="cuda")[:, None]).long()
    mask = lengths(50, 40, 30)
    call = lambda m: net(input_ids=ids, attention_mask=m).last_hidden_state
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            call(mask)
        torch.cuda.current_stream().wait_stream(side)
        call(mask)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            captured = call(mask)
        with torch.cuda.stream(side):   # the stream of the capture, which has not computed anything yet
            assert torch.isfinite(call(mask)).all()
        torch.cuda.synchronize()
        layer = net.encoder.layer[1].attention.self
        for step, n in enumerate(((50, 40, 30), (20, 50, 1), (7, 8, 50))):
            mask.copy_(lengths(*n))
            ids.copy_(torch.randint(0, 100, (3, 50), device="cuda"))
            if step == 2:
                layer.key_proj.weight.mul_(-1.5)
                net.encoder.rel_embeddings.weight.mul_(0.5)
            ref = call(lengths(*n))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(captured, ref), step
            assert torch.equal(call(mask), ref)


@pytest.mark.gpu
def test_projection_whose_weight_is_no_parameter():
    """Pruning leaves `weight` an attribute beside the parameter `weight_orig`."""
    from torch.nn.utils import prune

    att = _attention().eval()
    x, rel = torch.randn(1, 20, 128, device="cuda").to(torch.bfloat16), torch.randn(64, 128, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        ref = att(x, None, rel_embeddings=rel)[0]
        prune.identity(att.query_proj, "weight")
        assert torch.equal(att(x, None, rel_embeddings=rel)[0], ref)


@pytest.mark.gpu
def test_operands_of_another_device_or_size_are_refused():
    x, w, b = [torch.randn(*s, device="cuda").to(torch.bfloat16) for s in ((4, 64), (64, 64), (64,))]
    for bad in ((x, w.cpu(), b), (x, w, b.cpu()), (x, w, b[:32].contiguous())):
        with pytest.raises(RuntimeError):
            _lib.native.linear(*bad, True)
    q = torch.randn(1, 40, 2, 64, device="cuda").to(torch.bfloat16)
    pos = torch.randn(2, 64, 64, device="cuda").to(torch.bfloat16)
    lse = torch.zeros(40, 2, device="cuda")
    tail = (0.1, 32, 64, False, None, None)
    for bad in ((q, q, q, q, lse, q[:, :20], pos, pos), (q, q, q, q, lse[:20], q, pos, pos), (q, q, q, q, lse, q.float(), pos, pos),
                (q, q, q, q, lse, q, pos.cpu(), pos)):
        with pytest.raises(ValueError):
            _lib.native.attention_bwd(*bad, *tail)
    with pytest.raises(ValueError):
        _lib.native.attention_fwd(q, q.cpu(), q, pos, pos, None, None, 0.1, 32, 64, False, False, *([None] * 7), False, 0, 0, None, False, 0, None)


def _lets_others_run(call):
    """Whether another thread gets the interpreter during one of many calls.  Nobody asks for it back in the meantime (the switch
    interval is longer than the test), so it does only if the call itself lets go."""
    gate, ran = threading.Lock(), []
    gate.acquire()
    old = sys.getswitchinterval()
    sys.setswitchinterval(1000.0)
    other = threading.Thread(target=lambda: gate.acquire() and ran.append(1))
    other.start()
    gate.release()
    try:
        for _ in range(3000):
            call()
            if ran:
                return True
        return False
    finally:
        sys.setswitchinterval(old)
        other.join()


def _refused(call):
    def run():
        try:
            call()
        except RuntimeError:
            pass
    return run


def test_interpreter_lock_on_the_host():
    """The entries whose first part runs on CPU tensors, too: a projection, and (refused after it) the layers around one."""
    x, w, b = torch.randn(1, 64, 64), torch.randn(192, 64), torch.randn(192)
    norm, square = (b[:64], b[:64], 1e-7), (w[:64], b[:64])
    rest = (None, None, 1, 0.1, 0, 0, None, None)
    assert not _lets_others_run(lambda: _lib.native.untouched((), ()))
    assert _lets_others_run(lambda: _lib.native.linear(x, w, b, False))
    assert _lets_others_run(_refused(lambda: _lib.native.layer_attention(x, w, b, *rest, False)))
    assert _lets_others_run(_refused(lambda: _lib.native.encoder_layer(x, w, b, *rest, *square, *norm, *square, *square, *norm)))


@pytest.mark.gpu
def test_interpreter_lock_on_the_gpu():
    from flashdeberta_amd import ops

    g = lambda *s: torch.randn(*s, device="cuda").to(torch.bfloat16)
    q, pos, mask = g(1, 40, 2, 64), g(2, 64, 64), torch.ones(2, 40, device="cuda")
    kw = dict(position_buckets=32, max_relative_positions=64)
    out, lse = ops.disentangled_attention_fwd(q, q, q, pos, pos, return_lse=True, **kw)
    att, x, rel = _attention().train(), g(1, 40, 128), g(64, 128)
    leaf = q.clone().requires_grad_()
    cu = torch.tensor([0, 40], dtype=torch.int32, device="cuda")
    for call in (lambda: ops.disentangled_attention_fwd(q, q, q, pos, pos, **kw),
                 lambda: ops.disentangled_attention_fwd(q[0], q[0], q[0], pos, pos, cu_seqlens=cu, max_seqlen=40, **kw),   # asks Python on its way
                 lambda: ops.disentangled_attention_bwd(q, q, q, out, lse, q, pos, pos, **kw), lambda: ops.disentangled_attention(leaf, q, q, pos, pos, **kw),
                 lambda: att(x, None, rel_embeddings=rel), lambda: _lib.native.mask_bounds(mask), lambda: ops.quantize_e4m3_per_head(q),
                 lambda: ops.quantize_e4m3_per_head_pair(q, q)):
        assert _lets_others_run(call)
        torch.cuda.synchronize()


@pytest.mark.gpu
def test_threads_share_the_plans():
    """Forward and backward of layers of many lengths from several threads: the products' plans are made, found and launched by
    these threads and by autograd's own, which do not hold the GIL."""
    att = _attention().train()
    rel = torch.randn(64, 128, device="cuda").to(torch.bfloat16)
    xs = [torch.randn(1, n, 128, device="cuda").to(torch.bfloat16).requires_grad_() for n in range(33, 53)]

    def gradients(x):
        out = att(x, None, rel_embeddings=rel)[0]
        return torch.autograd.grad(out, [x, att.value_proj.bias], torch.ones_like(out))

    got, failed = {}, []

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                got[k] = [gradients(x) for x in xs[k % 2::2]]
                torch.cuda.current_stream().synchronize()
        except Exception as e:   # noqa: BLE001  (reported below, in the main thread)
            failed.append(e)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not failed, failed
    for k in range(4):
        for x, g in zip(xs[k % 2::2], got[k]):
            assert all(torch.equal(a, b) for a, b in zip(g, gradients(x)))


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,heads,dim", [(1, 1, 64), (1, 40, 64), (257, 3, 64), (511, 12, 32), (300, 17, 128), (16391, 12, 64), (40, 400, 64)])
def test_quantiser_walks_every_row(tokens, heads, dim):
    """Heads fewer and more than a workgroup has rows, tokens around a thread's eight; bytes and scales are whole, hence exact."""
    from flashdeberta_amd import quantize_e4m3_per_head_pair

    g = torch.Generator(device="cuda").manual_seed(tokens + heads)
    xs = [torch.randn(tokens, heads, dim + 8, device="cuda", generator=g).to(torch.bfloat16)[..., :dim] for _ in range(2)]
    y0, s0, y1, s1 = quantize_e4m3_per_head_pair(*xs)
    for x, y, s in ((xs[0], y0, s0), (xs[1], y1, s1)):
        scale = x.float().abs().amax(dim=(0, 2)).clamp_min(1e-12) / torch.tensor(448.0, device="cuda")   # a divisor on the GPU: a Python number would become a factor 1 / 448
        assert torch.equal(s, scale)
        assert torch.equal(y.view(torch.uint8), (x.float() / scale[:, None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8))
