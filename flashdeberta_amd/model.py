"""Drop-in attention module and the `_attn_implementation` switch.

Counterparts in the reference (src/flashdeberta/model.py):
  FlashDisentangledSelfAttention   :97-252   same constructor, parameters and forward signature
  DEBERTA_SELF_ATTENTION_CLASSES   :254-257  {"eager", "flash_attention_2"}
  FlashDebertaV2Model              :394-496  here a thin subclass of transformers' DebertaV2Model
The eager entry is transformers' own DisentangledSelfAttention, exactly as in the reference.
Differentiable like the reference's fixed-length op (padded batches included: they stay in the fixed layout
here); attention-probability dropout is not applied (nor is it on the reference's flash path: only the dropout
on the relative embeddings remains, model.py:159-160).
"""
import math
import threading

import torch
import torch.nn.functional as F
from torch.nn.modules import module as nn_module
from transformers.activations import GELUActivation
from transformers.models.deberta_v2.modeling_deberta_v2 import (
    DebertaV2Attention,
    DebertaV2Config,
    DebertaV2Encoder,
    DebertaV2Intermediate,
    DebertaV2Layer,
    DebertaV2Model,
    DebertaV2Output,
    DebertaV2SelfOutput,
    DisentangledSelfAttention,
)

from . import ops
from ._lib import native
from .padding import key_padding_mask, seq_bounds


# One remembered value, valid while the tensors it was computed from are the same objects, have not been written in
# place, still sit in the same storage with the same dtype on the same device, and `extra` compares equal; the tensors
# are held weakly: get(tensors, extra=None), put(tensors, value, extra=None).  Each of the last four streams has its own, and
# so has a graph that is being recorded: it computes what it needs anew, from the masks and weights as they are at a replay.
_Memo = native.Memo


def _seq_bounds_of(attention_mask, memo):
    """(seq_start, seq_len) of a mask.  Every layer of an encoder receives the same mask object, so the
    reductions run once per forward instead of once per layer: `memo` (a _Memo that the layers of a patched
    model share, see patch_model) holds the result for as long as the mask is the same object, unwritten and
    in place.  Nothing is stored on the caller's tensor and nothing is process-global."""
    hit = memo.get((attention_mask,))
    if hit is None:
        hit = native.mask_bounds(attention_mask)  # one launch; None where it does not read the mask (CPU, odd forms)
        if hit is None:
            hit = seq_bounds(key_padding_mask(attention_mask))[:2]
        memo.put((attention_mask,), hit)
    return hit


def _weight_and_bias(module):
    """A projection's parameters; a plain Linear's without nn.Module's attribute machinery (a quarter of a microsecond each)."""
    own = module._parameters
    if type(module) is torch.nn.Linear and "weight" in own and "bias" in own:  # pruning and weight_norm move them elsewhere
        return own["weight"], own["bias"]
    return module.weight, module.bias


def _kind(cls):
    """A class as native.untouched asks for it: with what it computes as long as nobody gives it another forward."""
    return cls, cls.forward


_LINEAR, _LAYER_NORM, _DROPOUT = _kind(torch.nn.Linear), _kind(torch.nn.LayerNorm), _kind(torch.nn.Dropout)


def _stands_in(modules, kinds):
    """Whether computing what these kinds of modules do without calling them is unseen by the program: native.untouched, and
    no hooks on all modules."""
    return native.untouched(modules, kinds) and not (nn_module._global_forward_hooks or nn_module._global_forward_pre_hooks
                                                     or nn_module._global_backward_hooks or nn_module._global_backward_pre_hooks)


_PROJECTIONS = "query_proj", "key_proj", "value_proj", "pos_key_proj", "pos_query_proj"
_PARTS = _LINEAR, _LINEAR, _LINEAR, _DROPOUT


class FlashDisentangledSelfAttention(DisentangledSelfAttention):
    """Same parameters as the eager module (query_proj, key_proj, value_proj[, pos_key_proj,
    pos_query_proj]), so `load_state_dict(eager.state_dict())` works (reference tests/attention.py:60).

    fp8_qk=True quantises Q, K and the projected relative embeddings to OCP e4m3 with per-head
    absmax scales before the kernel (bf16 inputs only).

    Outside training the three input projections run as one GEMM over the concatenated weights
    (a copy kept per module and stream, rebuilt when a parameter is replaced or written in place), and K_r / Q_r
    are remembered for as long as the relative embeddings handed in are the same tensor (an encoder
    patched by `patch_model` hands in the same tensor until its embedding table changes); both only
    while the projections are plain linear layers that nobody has hooked or given another forward."""

    # Projections of a few rows by the library's own kernels, which start sooner than hipBLASLt's but add up in another order;
    # off in a patched encoder, whose twelve layers turn one differing rounding of a 16-bit type into a percent.
    _own_products = True

    def __init__(self, config, fp8_qk=None):
        super().__init__(config)
        self.fp8_qk = bool(getattr(config, "fp8_qk", False)) if fp8_qk is None else bool(fp8_qk)
        self._qkv_memo, self._pos_memo, self._mask_memo, self._pos8_memo = _Memo(), _Memo(), _Memo(), _Memo()

    def _plain_projections(self):
        """Whether products with the projections' weights are all that the query, key and value projections do."""
        modules = self._modules
        return _stands_in((modules["query_proj"], modules["key_proj"], modules["value_proj"]), (_LINEAR, _LINEAR, _LINEAR))

    def _plain_parts(self):
        """The same for all parts: the projections of the relative embeddings and their dropout among them."""
        if not self.relative_attention:
            return self._plain_projections()
        modules = self._modules
        parts = modules["query_proj"], modules["key_proj"], modules["value_proj"], modules["pos_dropout"]
        if self.share_att_key:
            return _stands_in(parts, _PARTS)
        own = tuple(modules[n] for n in ("pos_key_proj", "pos_query_proj") if n in modules)
        return _stands_in(parts + own, _PARTS + (_LINEAR,) * len(own))

    def _recording(self, *inputs):
        """Whether autograd records what is computed from these tensors and the projections' weights, the ones that are read: a
        DataParallel replica holds its weights as plain attributes and has no parameters."""
        if not torch.is_grad_enabled():
            return False
        modules = self._modules
        weights = [p for n in _PROJECTIONS if n in modules for p in _weight_and_bias(modules[n])]
        return any(x is not None and x.requires_grad for x in (*inputs, *weights))

    def _fused_qkv(self):
        """Concatenated [3*H*D, hidden] weight and bias of the query, key and value projections (plain ones), None where only
        some have a bias."""
        modules = self._modules
        qw, qb = _weight_and_bias(modules["query_proj"])
        kw, kb = _weight_and_bias(modules["key_proj"])
        vw, vb = _weight_and_bias(modules["value_proj"])
        with_bias = qb is not None and kb is not None and vb is not None
        if not with_bias and not (qb is None and kb is None and vb is None):
            return None
        params = (qw, kw, vw, qb, kb, vb) if with_bias else (qw, kw, vw)
        hit = self._qkv_memo.get(params)
        if hit is None:
            with torch.no_grad():
                w = torch.cat([qw, kw, vw], dim=0)
                b = torch.cat([qb, kb, vb], dim=0) if with_bias else None
            hit = self._qkv_memo.put(params, (w, b))
        return hit

    def _qkv(self, hidden_states, query_states):
        """q, k, v as [B, L, H, D] views (reference model.py:147-149)."""
        B, L, _ = hidden_states.shape
        H, D = self.num_attention_heads, self.attention_head_size
        # the concatenated weights are a copy made outside autograd: only where nothing is being recorded
        fused = None if (self.training or query_states is not hidden_states or not self._plain_parts() or self._recording(hidden_states)) \
            else self._fused_qkv()
        if fused is not None:
            qkv = F.linear(hidden_states, fused[0], fused[1]).view(B, L, 3, H, D)
            return qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2]
        return (self.query_proj(query_states).view(B, L, H, D), self.key_proj(hidden_states).view(B, L, H, D),
                self.value_proj(hidden_states).view(B, L, H, D))

    def _pos_layers(self, rel_embeddings, plain=False, dropped=None):
        """K_r, Q_r as [H, 2S, D] views of the projected relative embeddings
        (reference model.py:159-177; the slice to 2S rows is transformers modeling_deberta_v2.py:295).
        plain: the caller knows that nobody has touched the parts and that nothing is recorded; dropped: what pos_dropout
        gave for these embeddings, if the caller has called it."""
        if not self.relative_attention or rel_embeddings is None:
            return None, None
        # the position projections exist only for the terms the module has (transformers :170-178)
        kproj = qproj = None
        modules = self._modules
        if "c2p" in self.pos_att_type:
            kproj = modules["key_proj" if self.share_att_key else "pos_key_proj"]
        if "p2c" in self.pos_att_type:
            qproj = modules["query_proj" if self.share_att_key else "pos_query_proj"]
        key = None
        dropout = modules["pos_dropout"]
        # a remembered K_r / Q_r must not carry an autograd graph, and depends on nothing but the embeddings and the weights
        if not self.training and (plain or self._plain_parts() and not self._recording(rel_embeddings)) and not (dropout.training and dropout.p > 0.0):
            key, terms = (rel_embeddings,), tuple(self.pos_att_type)
            for m in (kproj, qproj):
                if m is not None:
                    weight, bias = _weight_and_bias(m)
                    key += (weight, bias) if bias is not None else (weight,)
            hit = self._pos_memo.get(key, terms)
            if hit is not None:
                return hit
        H, D = self.num_attention_heads, self.attention_head_size
        span = self.pos_ebd_size
        rel = (dropout(rel_embeddings) if dropped is None else dropped)[0:2 * span]

        def heads(x):  # [2S, H*D] -> [H, 2S, D] without a copy
            return x.view(x.shape[0], H, D).transpose(0, 1)

        pos_key = heads(kproj(rel)) if kproj is not None else None
        pos_query = heads(qproj(rel)) if qproj is not None else None
        if key is not None:
            self._pos_memo.put(key, (pos_key, pos_query), terms)
        return pos_key, pos_query

    def _score_settings(self, pos_key, pos_query):
        """(sm_scale, position_buckets, max_relative_positions) of the operator (reference model.py:151-157)."""
        present = not self.relative_attention
        terms = 1 + ("c2p" in self.pos_att_type and (present or pos_key is not None)) + \
            ("p2c" in self.pos_att_type and (present or pos_query is not None))
        sm_scale = 1.0 / math.sqrt(self.attention_head_size * terms)
        return (sm_scale, self.position_buckets, self.max_relative_positions) if self.relative_attention else (sm_scale, 0, 0)

    def _bounds(self, attention_mask):
        """(seq_start, seq_len) of the batch.  The kernels take the real tokens of a row as one contiguous run and write
        zeros into the padded rows themselves; a row whose mask has a hole inside that run carries seq_len -1 and comes
        back as NaN in every position, so the unsupported mask cannot pass for a result (the eager module honours
        arbitrary masks)."""
        return (None, None) if attention_mask is None else _seq_bounds_of(attention_mask, self._mask_memo)

    def _native_args(self, attention_mask, rel_embeddings, hidden_states=None):
        """What follows the hidden states in a call of native.layer_attention, or None where that path does not serve:
        in training or while anything is recorded (the concatenated weights are a copy made outside autograd), under
        autocast, with FP8 operands, or with projections that are more than products with weights to concatenate."""
        if self.training or self.fp8_qk or torch.is_autocast_enabled():
            return None
        if not self._plain_parts() or self._recording(hidden_states, rel_embeddings):
            return None
        fused = self._fused_qkv()
        if fused is None:
            return None
        pos_key, pos_query = self._pos_layers(rel_embeddings, plain=True)
        return (*fused, pos_key, pos_query, self.num_attention_heads, *self._score_settings(pos_key, pos_query), *self._bounds(attention_mask))

    def _trains_as_one_node(self):
        """Whether native.layer_node computes what the module does, step by step: plain projections shared with the tables, both
        position terms, nothing that has to see the projections' own calls (hooks, a forward of their own) or cast their operands
        (autocast)."""
        if not (self.relative_attention and self.share_att_key and not self.fp8_qk and "c2p" in self.pos_att_type and "p2c" in self.pos_att_type) \
                or torch.is_autocast_enabled() or torch.compiler.is_compiling():
            return False
        return self._plain_projections()

    def forward(self, hidden_states, attention_mask, output_attentions=False, query_states=None,
                relative_pos=None, rel_embeddings=None):
        """-> (context [B, L, H*D], None).  `relative_pos` is ignored: the bucketed relative
        position is an integer table inside the kernel.  Attention probabilities are never
        materialised, so `output_attentions` yields None like the reference (model.py:252)."""
        # Under autograd the fused op is one node: differentiable in fp32 / bf16 / fp16 (the reference's
        # FlashAttentionDisentangled, flash_attention.py:1032-1086); with FP8 operands its backward raises.
        if query_states is None:
            query_states = hidden_states
        B, L, _ = hidden_states.shape
        H, D = self.num_attention_heads, self.attention_head_size
        args = self._native_args(attention_mask, rel_embeddings, hidden_states) if query_states is hidden_states else None
        if args is not None:
            return native.layer_attention(hidden_states, *args, self._own_products), None
        seq_start, seq_len = self._bounds(attention_mask)
        rel = None
        if query_states is hidden_states and rel_embeddings is not None and self._trains_as_one_node():
            sm_scale, buckets, max_distance = self._score_settings(rel_embeddings, rel_embeddings)
            modules = self._modules
            rel = self.pos_dropout(rel_embeddings)
            ctx = native.layer_node(hidden_states, rel, *[p for n in ("query_proj", "key_proj", "value_proj") for p in _weight_and_bias(modules[n])],
                                    H, sm_scale, buckets, max_distance, seq_start, seq_len)
            if ctx is not None:
                return ctx, None
        pos_key, pos_query = self._pos_layers(rel_embeddings, dropped=rel)
        sm_scale, buckets, max_distance = self._score_settings(pos_key, pos_query)

        q, k, v = self._qkv(hidden_states, query_states)
        kw = {}
        if self.fp8_qk:
            if q.dtype != torch.bfloat16:
                raise ValueError("fp8_qk needs bfloat16 activations")
            # q and k of the layer in one set of launches; K_r / Q_r likewise, and remembered for as long as the
            # projected relative embeddings are the same tensors (outside training they are, see _pos_layers)
            q, kw["q_scale"], k, kw["k_scale"] = ops.quantize_e4m3_per_head_pair(q, k)
            pos = tuple(x for x in (pos_key, pos_query) if x is not None)
            hit = self._pos8_memo.get(pos) if pos else None
            if hit is None and pos:
                if len(pos) == 2:
                    k8, ks, q8, qs = ops.quantize_e4m3_per_head_pair(pos_key.transpose(0, 1), pos_query.transpose(0, 1))
                    hit = (k8.transpose(0, 1), ks, q8.transpose(0, 1), qs)
                else:
                    y, sc = ops.quantize_e4m3_per_head(pos[0].transpose(0, 1))
                    hit = (y.transpose(0, 1), sc, None, None) if pos_key is not None else (None, None, y.transpose(0, 1), sc)
                if not (torch.is_grad_enabled() and any(x.requires_grad for x in pos)):
                    self._pos8_memo.put(pos, hit)
            if pos:
                pos_key, pos_key_scale, pos_query, pos_query_scale = hit
                if pos_key is not None:
                    kw["pos_key_scale"] = pos_key_scale
                if pos_query is not None:
                    kw["pos_query_scale"] = pos_query_scale

        ctx = ops.disentangled_attention(
            q, k, v, pos_key, pos_query, sm_scale=sm_scale,
            position_buckets=buckets, max_relative_positions=max_distance, seq_start=seq_start, seq_len=seq_len, **kw)
        return (ctx.view(B, L, H * D), None)


DEBERTA_SELF_ATTENTION_CLASSES = {
    "eager": DisentangledSelfAttention,
    "flash_attention_2": FlashDisentangledSelfAttention,
}


# the parts of a layer that its one native call takes the place of, in the order FlashDebertaV2Layer._native_args names them
_LAYER_PARTS = (*(_kind(c) for c in (DebertaV2Attention, DebertaV2Intermediate, DebertaV2Output, FlashDisentangledSelfAttention, DebertaV2SelfOutput,
                                     GELUActivation)), *(_LINEAR,) * 3, *(_LAYER_NORM,) * 2, *(_DROPOUT,) * 2)


class FlashDebertaV2Layer(DebertaV2Layer):
    """transformers' encoder layer whose inference in a 16-bit type is one native call (native.encoder_layer): the same
    projections, attention, GELU and post-norms, with the same bits, without a module call per step.
    Anything else -- training, recording, autocast, hooks on any part, a part with a forward of its own or of another class
    (adapters, quantised projections, another activation), a dropout that is on -- takes transformers' own forward.  Instances are
    made by `patch_model`."""

    def _native_args(self, hidden_states, attention_mask, rel_embeddings):
        if self.training or torch.is_grad_enabled() or hidden_states.dtype not in (torch.bfloat16, torch.float16) or not hidden_states.is_cuda \
                or torch.compiler.is_compiling():
            return None
        own = self._modules
        attention, intermediate, output = own["attention"], own["intermediate"], own["output"]
        if type(attention) is not DebertaV2Attention or type(intermediate) is not DebertaV2Intermediate or type(output) is not DebertaV2Output:
            return None
        att, att_out = attention._modules["self"], attention._modules["output"]
        if type(att_out) is not DebertaV2SelfOutput:
            return None
        act = intermediate._modules.get("intermediate_act_fn")
        linears = att_out._modules["dense"], intermediate._modules["dense"], output._modules["dense"]
        norms = att_out._modules["LayerNorm"], output._modules["LayerNorm"]
        dropouts = att_out._modules["dropout"], output._modules["dropout"]
        if not _stands_in((attention, intermediate, output, att, att_out, act, *linears, *norms, *dropouts), _LAYER_PARTS):
            return None
        if act.act is not F.gelu or any(m.training and m.p > 0.0 for m in dropouts):
            return None
        shape, dtype = hidden_states.shape[-1:], hidden_states.dtype
        if any(m.weight.dtype != dtype for m in linears):
            return None
        if any(m.normalized_shape != shape or m.bias is None or m.weight is None or m.weight.dtype != dtype for m in norms):
            return None
        args = att._native_args(attention_mask, rel_embeddings)
        if args is None:
            return None
        (ow, ob), (uw, ub), (dw, db) = [_weight_and_bias(m) for m in linears]
        n1, n2 = norms
        return (*args, ow, ob, n1.weight, n1.bias, n1.eps, uw, ub, dw, db, n2.weight, n2.bias, n2.eps)

    def forward(self, hidden_states, attention_mask, query_states=None, relative_pos=None, rel_embeddings=None, output_attentions=False):
        if query_states is None or query_states is hidden_states:
            args = self._native_args(hidden_states, attention_mask, rel_embeddings)
            if args is not None:
                return native.encoder_layer(hidden_states, *args), None
        return super().forward(hidden_states, attention_mask, query_states=query_states, relative_pos=relative_pos,
                               rel_embeddings=rel_embeddings, output_attentions=output_attentions)


_forwarding = threading.local()   # the encoder whose forward this thread is in


class FlashDebertaV2Encoder(DebertaV2Encoder):
    """transformers' encoder minus work the fused attention never reads: with `_fdb_skip_dense` it builds
    neither the [1, L, L] int64 relative-position tensor nor the [B, 1, L, L] mask (transformers
    modeling_deberta_v2.py:601-626), and outside training it hands the layers one relative-embedding tensor
    object for as long as the table and its LayerNorm are unchanged, so that each layer's K_r / Q_r stay
    valid from forward to forward.  A forward that autograd records (an eval model that is fine-tuned) computes
    the tensor with its graph, each time.  Instances are made by `patch_model`, which switches the class of an
    existing encoder."""

    _fdb_skip_dense = True

    def forward(self, *args, **kwargs):
        outer = getattr(_forwarding, "encoder", None)
        _forwarding.encoder = self
        try:
            return super().forward(*args, **kwargs)
        finally:
            _forwarding.encoder = outer

    def get_rel_pos(self, hidden_states, query_states=None, relative_pos=None):
        if self._fdb_skip_dense:
            return relative_pos
        return super().get_rel_pos(hidden_states, query_states, relative_pos)

    def get_attention_mask(self, attention_mask):
        if self._fdb_skip_dense:
            return attention_mask
        return super().get_attention_mask(attention_mask)

    def get_rel_embedding(self):
        if self.training or not self.relative_attention:
            return super().get_rel_embedding()
        memo = self.__dict__.get("_fdb_rel_memo")
        if memo is None:
            memo = self._fdb_rel_memo = _Memo()
        norm = self.LayerNorm if "layer_norm" in self.norm_rel_ebd else None
        key = (self.rel_embeddings.weight,) + (() if norm is None else tuple(p for p in (norm.weight, norm.bias) if p is not None))
        recorded = getattr(_forwarding, "encoder", None) is self and torch.is_grad_enabled() and any(p.requires_grad for p in key)
        if recorded or not (norm is None or _stands_in((norm,), (_LAYER_NORM,))):
            return super().get_rel_embedding()
        hit = memo.get(key)
        if hit is None:
            with torch.no_grad():
                hit = memo.put(key, super().get_rel_embedding())
        return hit


def patch_model(model, attn_implementation="flash_attention_2", fp8_qk=False, skip_dense_position_tensors=True):
    """Swap every `layer.attention.self` of a transformers DebertaV2 model (bare or with a head)
    for the class the key selects, keeping the weights.  With skip_dense_position_tensors the
    encoder also stops building the [1, L, L] int64 relative-position tensor and the [B, 1, L, L]
    mask (transformers modeling_deberta_v2.py:601-626), which the fused path never reads."""
    cls = DEBERTA_SELF_ATTENTION_CLASSES[attn_implementation]
    encoder = None
    for mod in model.modules():
        if mod.__class__.__name__ == "DebertaV2Encoder" or hasattr(mod, "rel_embeddings") and hasattr(mod, "layer"):
            encoder = mod
            break
    if encoder is None:
        raise ValueError("no DebertaV2 encoder found in %s" % type(model).__name__)
    config = model.config
    mask_memo = _Memo()  # the layers of one model see the same mask object: its bounds are derived once per forward
    for layer in encoder.layer:
        old = layer.attention.self
        if type(old) is cls:
            if cls is FlashDisentangledSelfAttention:
                old._mask_memo = mask_memo
                old._own_products = False
            continue
        new = cls(config, fp8_qk=fp8_qk) if cls is FlashDisentangledSelfAttention else cls(config)
        new.load_state_dict(old.state_dict())
        p = next(old.parameters())
        new.to(device=p.device, dtype=p.dtype)
        new.train(old.training)
        if cls is FlashDisentangledSelfAttention:
            new._mask_memo = mask_memo
            new._own_products = False
        layer.attention.self = new
    flash = cls is FlashDisentangledSelfAttention
    for layer in encoder.layer:
        if flash and type(layer) is DebertaV2Layer:
            layer.__class__ = FlashDebertaV2Layer
        elif not flash and type(layer) is FlashDebertaV2Layer:
            layer.__class__ = DebertaV2Layer
    # The encoder-side shortcuts live in a subclass that differs from transformers' encoder in three methods
    # only; switching the instance's class keeps copies and pickles of the model working.
    if flash and type(encoder) in (DebertaV2Encoder, FlashDebertaV2Encoder):
        encoder.__class__ = FlashDebertaV2Encoder
        encoder._fdb_skip_dense = bool(skip_dense_position_tensors)
        encoder._fdb_rel_memo = _Memo()
    elif type(encoder) is FlashDebertaV2Encoder:
        encoder.__class__ = DebertaV2Encoder
    return model


class FlashDebertaV2Model(DebertaV2Model):
    """DebertaV2Model whose attention follows `config._attn_implementation` in
    {"eager", "flash_attention_2"}; unset means "flash_attention_2", the reference's default
    (model.py:61-62).  transformers' own check would treat "flash_attention_2" as a request for
    the flash-attn package, so the two keys are resolved here instead."""

    def _check_and_adjust_attn_implementation(self, attn_implementation, is_init_check=False, **kwargs):
        if attn_implementation is None:
            return "flash_attention_2"
        if attn_implementation in DEBERTA_SELF_ATTENTION_CLASSES:
            return attn_implementation
        raise ValueError("attn_implementation must be one of %s, got %r"
                         % (sorted(DEBERTA_SELF_ATTENTION_CLASSES), attn_implementation))

    def __init__(self, config):
        super().__init__(config)
        patch_model(self, self.config._attn_implementation, fp8_qk=bool(getattr(config, "fp8_qk", False)))


__all__ = ["FlashDisentangledSelfAttention", "DEBERTA_SELF_ATTENTION_CLASSES", "FlashDebertaV2Model",
           "FlashDebertaV2Encoder", "FlashDebertaV2Layer", "DebertaV2Config", "patch_model"]
