"""Performance cases of the disentangled attention: what a program built on this package has it compute.

Each case is a dict of plain values; `path` says which public entry point it goes through:

  layer        FlashDisentangledSelfAttention, inference (projections + attention, right-padded batches with a mask)
  encoder      FlashDebertaV2Model, inference (a whole v3-base encoder)
  attention    disentangled_attention_fwd on [B, L, H, D] tensors in bf16, fp16 or fp32
  packed       flash_attention_with_disentangled_varlen on [T, H, D] tensors
  fp8          quantize_e4m3_per_head_pair of q and k, then disentangled_attention_fwd on the e4m3 operands
  train_layer  FlashDisentangledSelfAttention, forward and backward (gradients of the input, of the relative embeddings
               and of every weight)
  train        flash_attention_with_disentangled, forward and backward ([B, H, L, D] as that operator takes them)

The relative positions are v3's throughout: 256 buckets over 512 positions, both position terms.
"""
import math
import random

import torch

from flashdeberta_amd import (
    DebertaV2Config,
    FlashDebertaV2Model,
    FlashDisentangledSelfAttention,
    disentangled_attention_fwd,
    flash_attention_with_disentangled,
    flash_attention_with_disentangled_varlen,
    quantize_e4m3_per_head,
    quantize_e4m3_per_head_pair,
)

BUCKETS, MAX_DISTANCE = 256, 512
TABLE = 2 * BUCKETS  # rows of K_r and of Q_r
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # one short query at an interactive service: latency, launches and host time are everything
        dict(name="layer_1x24_bf16", path="layer", dtype="bf16", batch=1, length=24, heads=12, padded=False),
        # a batch of short texts for classification, padded to the longest
        dict(name="layer_32x128_padded_bf16", path="layer", dtype="bf16", batch=32, length=128, heads=12, padded=True),
        # the whole encoder at the usual training length, as embedding and tagging jobs run it
        dict(name="encoder_8x512_padded_bf16", path="encoder", dtype="bf16", batch=8, length=512, heads=12, layers=12, padded=True),
        # a few documents of a length nothing is tuned for
        dict(name="attention_3x777_fp16", path="attention", dtype="fp16", batch=3, length=777, heads=12, dim=64),
        # long documents, a full batch: the shape the headline figure is quoted on
        dict(name="attention_8x4096_bf16", path="attention", dtype="bf16", batch=8, length=4096, heads=12, dim=64),
        # one long document through the large model
        dict(name="attention_1x4096_h16_bf16", path="attention", dtype="bf16", batch=1, length=4096, heads=16, dim=64),
        # full precision, one sequence: parity runs and small exports
        dict(name="attention_1x512_fp32", path="attention", dtype="fp32", batch=1, length=512, heads=12, dim=64),
        # a packed batch of documents of very different lengths
        dict(name="packed_64_bf16", path="packed", dtype="bf16", sequences=64, shortest=32, longest=2048, heads=12, lengths_seed=1004),
        # very long documents with e4m3 scores, quantised on the way in
        dict(name="fp8_4x8192", path="fp8", dtype="fp8", batch=4, length=8192, heads=12),
        # fine-tuning: one layer's share of a step on a padded batch
        dict(name="train_layer_8x512_padded_bf16", path="train_layer", dtype="bf16", batch=8, length=512, heads=12, padded=True),
        # training on documents of an odd length
        dict(name="train_2x1501_fp16", path="train", dtype="fp16", batch=2, length=1501, heads=12),
        # training on long documents
        dict(name="train_8x4096_bf16", path="train", dtype="bf16", batch=8, length=4096, heads=12),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch(rng, length, most_tokens, most):
    return max(1, min(most, _log_int(rng, 1, max(1, min(most, most_tokens // length)))))


def draw(rng):
    path = rng.choice(["layer", "layer", "encoder", "attention", "attention", "attention", "packed", "fp8", "train_layer", "train_layer",
                       "train", "train"])
    heads = rng.choice([12, 12, 16])
    half = rng.choice(["bf16", "bf16", "fp16"])
    if path == "layer":
        length = _log_int(rng, 8, 512)
        return dict(path=path, dtype=half, batch=_batch(rng, length, 8192, 64), length=length, heads=rng.choice([6, 12, 16]),
                    padded=rng.random() < 0.7)
    if path == "encoder":
        length = _log_int(rng, 16, 512)
        return dict(path=path, dtype=half, batch=_batch(rng, length, 4096, 32), length=length, heads=12, layers=12, padded=rng.random() < 0.7)
    if path == "attention":
        if rng.random() < 0.3:
            length = _log_int(rng, 48, 2048)
            dim = rng.choice([64, 64, 128])
            return dict(path=path, dtype="fp32", batch=_batch(rng, length, 4096, 8), length=length, heads=heads if dim == 64 else 8, dim=dim)
        length = _log_int(rng, 64, 4096)
        return dict(path=path, dtype=half, batch=_batch(rng, length, 32768, 64), length=length, heads=heads, dim=64)
    if path == "packed":
        shortest, longest = _log_int(rng, 16, 64), _log_int(rng, 256, 2048)
        return dict(path=path, dtype=half, sequences=_log_int(rng, 4, 64), shortest=shortest, longest=longest, heads=12,
                    lengths_seed=rng.randrange(1 << 20))
    if path == "fp8":
        length = _log_int(rng, 512, 8192)
        return dict(path=path, dtype="fp8", batch=_batch(rng, length, 32768, 16), length=length, heads=12)
    if path == "train_layer":
        length = _log_int(rng, 32, 512)
        return dict(path=path, dtype=half, batch=_batch(rng, length, 8192, 64), length=length, heads=heads, padded=rng.random() < 0.7)
    length = _log_int(rng, 256, 4096)
    return dict(path=path, dtype=half, batch=_batch(rng, length, 16384, 16), length=length, heads=heads)


def _config(case):
    width = 64 * case["heads"]
    return DebertaV2Config(vocab_size=32000, hidden_size=width, num_hidden_layers=case.get("layers", 1), num_attention_heads=case["heads"],
                           intermediate_size=4 * width, relative_attention=True, pos_att_type="p2c|c2p", position_buckets=BUCKETS,
                           share_att_key=True, norm_rel_ebd="layer_norm", position_biased_input=False, max_position_embeddings=MAX_DISTANCE,
                           hidden_dropout_prob=0.0, attention_probs_dropout_prob=0.0)


def _row_lengths(case):
    """Real tokens per row of a padded batch: between a quarter of the longest row and all of it."""
    if not case["padded"]:
        return [case["length"]] * case["batch"]
    rng = random.Random(case["batch"] * 8191 + case["length"])
    full = case["length"]
    return [full] + [rng.randint(max(1, full // 4), full) for _ in range(case["batch"] - 1)]


def _packed_lengths(case):
    rng = random.Random(case["lengths_seed"])
    return [_log_int(rng, case["shortest"], case["longest"]) for _ in range(case["sequences"])]


def _mask(case):
    if not case["padded"]:
        return None
    lengths = torch.tensor(_row_lengths(case), device="cuda")
    return (torch.arange(case["length"], device="cuda") < lengths[:, None]).long()


def prepare(case, seed):
    """The program's inputs and what it keeps between calls (weights, tables).  Activations are unit normal, as they leave
    a layer norm; weights come from the model's own initialisation."""
    path = case["path"]
    dtype = DTYPES.get(case["dtype"], torch.bfloat16)
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).to(dtype)

    s = {"path": path}
    if path in ("layer", "train_layer", "encoder"):
        config = _config(case)
        torch.manual_seed(seed)
        with torch.device("cuda"):
            module = FlashDebertaV2Model(config) if path == "encoder" else FlashDisentangledSelfAttention(config)
        s["module"] = module.to(dtype).train(path == "train_layer")
        s["mask"] = _mask(case)
        if path == "encoder":
            s["ids"] = torch.randint(0, config.vocab_size, (case["batch"], case["length"]), device="cuda", generator=gen)
            return s
        s["x"] = normal(case["batch"], case["length"], config.hidden_size)
        s["rel"] = normal(TABLE, config.hidden_size)
        if path == "train_layer":
            s["grad"] = normal(*s["x"].shape)
            s["leaves"] = [s["x"].requires_grad_(), s["rel"].requires_grad_(), *s["module"].parameters()]
        return s
    heads, dim = case["heads"], case.get("dim", 64)
    if path == "packed":
        lengths = _packed_lengths(case)
        shape = (sum(lengths), heads, dim)
        ends = [0]
        for n in lengths:
            ends.append(ends[-1] + n)
        s["ends"], s["longest"] = torch.tensor(ends, dtype=torch.int32, device="cuda"), max(lengths)
    elif path == "train":
        shape = (case["batch"], heads, case["length"], dim)
    else:
        shape = (case["batch"], case["length"], heads, dim)
    s["scale"] = 1.0 / math.sqrt(3 * dim)
    s["q"], s["k"], s["v"] = normal(*shape), normal(*shape), normal(*shape)
    s["pos_key"], s["pos_query"] = normal(heads, TABLE, dim), normal(heads, TABLE, dim)
    if path == "fp8":
        for name in ("pos_key", "pos_query"):  # quantised once, like weights
            y, s[name + "_scale"] = quantize_e4m3_per_head(s[name].transpose(0, 1))
            s[name] = y.transpose(0, 1)
    if path == "train":
        s["leaves"] = [s[n].requires_grad_() for n in ("q", "k", "v", "pos_key", "pos_query")]
        s["grad"] = normal(*shape)
    return s


def run(s):
    path = s["path"]
    if path == "layer":
        with torch.no_grad():
            return s["module"](s["x"], s["mask"], rel_embeddings=s["rel"])[0]
    if path == "encoder":
        with torch.no_grad():
            return s["module"](input_ids=s["ids"], attention_mask=s["mask"]).last_hidden_state
    if path == "attention":
        return disentangled_attention_fwd(s["q"], s["k"], s["v"], s["pos_key"], s["pos_query"], position_buckets=BUCKETS,
                                          max_relative_positions=MAX_DISTANCE)
    if path == "packed":
        return flash_attention_with_disentangled_varlen(s["q"], s["k"], s["v"], s["pos_key"], s["pos_query"], s["ends"], s["ends"],
                                                        s["longest"], s["longest"], sm_scale=s["scale"], position_buckets=BUCKETS,
                                                        max_relative_distance=MAX_DISTANCE)
    if path == "fp8":
        q, q_scale, k, k_scale = quantize_e4m3_per_head_pair(s["q"], s["k"])
        return disentangled_attention_fwd(q, k, s["v"], s["pos_key"], s["pos_query"], q_scale=q_scale, k_scale=k_scale,
                                          pos_key_scale=s["pos_key_scale"], pos_query_scale=s["pos_query_scale"],
                                          position_buckets=BUCKETS, max_relative_positions=MAX_DISTANCE)
    if path == "train_layer":
        out = s["module"](s["x"], s["mask"], rel_embeddings=s["rel"])[0]
    else:
        out = flash_attention_with_disentangled(s["q"], s["k"], s["v"], s["pos_key"], s["pos_query"], sm_scale=s["scale"],
                                                position_buckets=BUCKETS, max_relative_distance=MAX_DISTANCE)
    return (out.detach(), *torch.autograd.grad(out, s["leaves"], s["grad"]))


def work(case):
    """Bytes and operations of one pass that no implementation does without: every input read and every output written
    once, the matrix products of the projections over all rows, and the attention's over the real tokens -- two products
    of length x length per head and one of each operand with the table rows its relative positions reach.  A backward pass
    doubles the projections and takes 2.5 times the attention's products."""
    path, heads, dim = case["path"], case["heads"], case.get("dim", 64)
    if path == "packed":
        lengths = _packed_lengths(case)
        rows = sum(lengths)
    else:
        lengths = _row_lengths(case) if "padded" in case else [case["length"]] * case["batch"]
        rows = case["batch"] * case["length"]
    attention = sum(4 * n * n * dim + 4 * n * min(TABLE, 2 * n - 1) * dim for n in lengths) * heads
    width = heads * dim
    size = BYTES.get(case["dtype"], 2)
    tensor, table = rows * width * size, TABLE * width * size
    weights = 3 * width * width * size
    if path == "layer":
        return {"bytes": 2 * tensor + 2 * table + weights, "flops": attention + 6 * rows * width * width}
    if path == "encoder":
        per_layer = attention + 24 * rows * width * width
        return {"bytes": tensor + case["layers"] * 4 * weights + rows * (8 + width * size), "flops": case["layers"] * per_layer}
    if path == "train_layer":
        return {"bytes": 4 * tensor + 2 * table + 2 * weights, "flops": 3.5 * attention + 18 * (rows + TABLE) * width * width}
    if path == "train":
        return {"bytes": 8 * tensor + 4 * table, "flops": 3.5 * attention}
    if path == "fp8":
        return {"bytes": 4 * tensor + table, "flops": attention}
    return {"bytes": 4 * tensor + 2 * table, "flops": attention}


def tolerance(case):
    if case["path"] == "fp8":
        return {"rel": 2e-2}
    if case["path"].startswith("train"):  # the backward rounds the probabilities and the score gradients on its way
        return {"rel": {"bf16": 1.5e-2, "fp16": 3e-3}[case["dtype"]]}
    return {"rel": {"bf16": 1e-2, "fp16": 2e-3, "fp32": 1e-5}[case["dtype"]]}
