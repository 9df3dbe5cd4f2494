"""Padded batches whose workgroups are dealt by the lengths of their sequences (padded_map in csrc/fdb_device.h): the bits of the same sequences in a batch of more
than 64, which is dealt in the plain order."""
import ctypes
import random

import pytest
import torch

from flashdeberta_amd import _lib, ops

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


def _call(x, starts, lens, more, grads, causal=False):
    """Forward (and backward) of the batch and, `more`, as many empty sequences behind it."""
    q, k, v, pk, pq, dout = x
    wide = lambda t: torch.cat([t, torch.zeros(more, *t.shape[1:], device="cuda", dtype=t.dtype)]) if more else t
    vec = lambda t: torch.tensor(list(t) + [0] * more, dtype=torch.int32, device="cuda")
    kw = dict(position_buckets=32, max_relative_positions=64, causal=causal, seq_start=vec(starts) if any(starts) else None, seq_len=vec(lens))
    q, k, v, dout = [wide(t) for t in (q, k, v, dout)]
    hold = torch.full((q.numel() * 4,), float("nan"), device="cuda", dtype=q.dtype)
    del hold   # what the outputs are given
    out, lse = ops.disentangled_attention_fwd(q, k, v, pk, pq, return_lse=True, **kw)
    n = out.shape[0] - more
    res = [out[:n], lse.view(out.shape[0], -1)[:n]]
    if grads:
        res += [g[:n] for g in ops.disentangled_attention_bwd(q, k, v, out, lse, dout, pk, pq, **kw)[:3]]
    return [t.nan_to_num(nan=12345.0) for t in res]


@pytest.mark.parametrize("causal", [False, True], ids=["all", "causal"])
@pytest.mark.parametrize("kind", ["ragged", "equal", "left", "odd"])
@pytest.mark.parametrize("B,L,H,dtype", [(2, 600, 32, torch.bfloat16), (64, 130, 3, torch.float16), (33, 129, 5, torch.bfloat16), (23, 385, 4, torch.bfloat16), (9, 1100, 6, torch.float16),
                                         (40, 200, 4, torch.float32), (64, 520, 8, torch.bfloat16)])   # the last: the backward's roles as two launches
def test_bits_of_the_plain_order(B, L, H, dtype, kind, causal):
    g = torch.Generator(device="cuda").manual_seed(B + L)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)
    x = rnd(B, L, H, 64), rnd(B, L, H, 64), rnd(B, L, H, 64), rnd(H, 64, 64), rnd(H, 64, 64), rnd(B, L, H, 64)
    starts, lens = _bounds(kind, B, L)
    assert B * ((L + 127) // 128) * H > 256
    grads = dtype != torch.float32 and min(lens) >= 0
    for a, b in zip(_call(x, starts, lens, 0, grads, causal), _call(x, starts, lens, 65, grads, causal)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kind", ["ragged", "left", "odd"])
@pytest.mark.parametrize("B,L,H,D,dtype,more", [
    (12, 400, 10, 32, torch.bfloat16, {}), (10, 900, 6, 32, torch.float16, {}), (9, 800, 7, 32, torch.bfloat16, dict(causal=True)),   # near launch alone, and with a far one
    (20, 300, 8, 128, torch.bfloat16, {}), (9, 700, 8, 128, torch.float16, dict(causal=True)), (30, 200, 8, 128, torch.float32, {}), (20, 260, 8, 32, torch.float32, dict(causal=True)),
    (14, 500, 8, 64, torch.float16, dict(single_kernel=True)), (14, 500, 8, 64, torch.float32, dict(causal=True)),
    (20, 380, 8, 64, "e4m3", {}), (12, 1100, 5, 64, "e4m3", {}), (12, 1000, 5, 64, "e4m3", dict(causal=True)), (12, 500, 9, 128, "e4m3", {})])
def test_bits_of_the_plain_order_in_every_kernel(B, L, H, D, dtype, more, kind):
    """The forward of the other head_dims, types and launches."""
    fp8 = dtype == "e4m3"
    g = torch.Generator(device="cuda").manual_seed(B + L)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(torch.bfloat16 if fp8 else dtype)
    q, k, v, pk, pq = rnd(B, L, H, D), rnd(B, L, H, D), rnd(B, L, H, D), rnd(H, 64, D), rnd(H, 64, D)
    kw = dict(position_buckets=32, max_relative_positions=64, return_lse=not more.get("single_kernel"), **more)
    if fp8:
        q, kw["q_scale"], k, kw["k_scale"] = ops.quantize_e4m3_per_head_pair(q, k)
        (pk, kw["pos_key_scale"]), (pq, kw["pos_query_scale"]) = [(y.transpose(0, 1), z) for y, z in (ops.quantize_e4m3_per_head(t.transpose(0, 1)) for t in (pk, pq))]
    starts, lens = _bounds(kind, B, L)
    assert B * ((L + 127) // 128) * H >= 400   # no shares of the keys either way
    got = []
    for extra in (0, 65):
        wide = lambda t: torch.cat([t.view(torch.uint8), torch.zeros(extra, *t.view(torch.uint8).shape[1:], device="cuda", dtype=torch.uint8)]).view(t.dtype)
        vec = lambda t: torch.tensor(list(t) + [0] * extra, dtype=torch.int32, device="cuda")
        res = ops.disentangled_attention_fwd(wide(q), wide(k), wide(v), pk, pq, seq_start=vec(starts) if any(starts) else None, seq_len=vec(lens), **kw)
        out, lse = res if kw["return_lse"] else (res, None)
        got.append([out[:B].nan_to_num(nan=12345.0)] + ([] if lse is None else [lse.view(B + extra, -1)[:B].nan_to_num(nan=12345.0)]))
    for a, b in zip(*got):
        assert torch.equal(a, b)


class _BwdArgs(ctypes.Structure):   # fdb_attn_bwd_tables_args of include/fdb.h
    _fields_ = [(n, ctypes.c_void_p) for n in "q k v dout out pos_key pos_query dq dk dv d_pos_key d_pos_query lse seq_start seq_len delta_lut workspace".split()] + \
        [(f"{t}_stride_{x}", ctypes.c_int64) for t in "q k v do out dq dk dv".split() for x in "bth"] + [(f"{t}_stride_{x}", ctypes.c_int64) for t in "pk pq dp".split() for x in "hr"] + \
        [(n, ctypes.c_int32) for n in "batch heads head_dim seqlen att_span lut_radius dtype causal".split()] + [("sm_scale", ctypes.c_float)]


def _plain_order(B, H, tiles, causal, keys):
    """block_map: the (sequence, head) groups of an L2's share at a time, a group on one XCD, a tile of all of them before the next."""
    most, out = 8 * (96 // tiles if tiles < 96 else 1), []
    for first in range(0, B * H, most):
        here = min(B * H - first, most)
        for m in range(tiles * here):
            t, i = divmod(m, here)
            n = first * tiles + m
            g = first + (n % 8 | i & ~7 if i < here & ~7 else i)
            if causal:
                t = t if keys else tiles - 1 - t
            else:
                t = tiles - 1 - t
                t = tiles - 1 - t // 2 if t % 2 else t // 2
            out.append((g // H, t, g % H))
    return out


def _order_by_length(lens, H, tiles, causal, keys):
    """The sequences with the most tiles first, those of a number of tiles as a batch of their own; causal: the highest tile of all sequences first, of key tiles the one as
    far from the text's end as the query tile of that turn is from its beginning.  Then the tiles of padding."""
    order = sorted(range(len(lens)), key=lambda b: (-((lens[b] + 31) // 32), b))
    of = lambda b: (lens[b] + 127) // 128
    if causal:
        real = [(b, of(b) - 1 - t if keys else t, h) for t in reversed(range(tiles)) for b in order if of(b) > t for h in range(H)]
    else:
        real = []
        for n in range(tiles, 0, -1):
            alike = [b for b in order if of(b) == n]
            real += [(alike[x], t, h) for x, t, h in _plain_order(len(alike), H, n, False, keys)]
    return real + [(b, t, h) for t in range(tiles) for b in order if of(b) <= t for h in range(H)]


@pytest.mark.parametrize("lens,L,H,causal", [
    ([300, 300, 300], 300, 30, False), ([512] * 8, 512, 12, True), ([400, 384, 512, 384], 512, 17, False),   # a mask that hides little or nothing
    ([400, 383, 512, 384], 512, 17, False), ([120, 128, 33, 0, 97] * 4, 128, 7, False), ([300, 700, -1, 699, 64, 0, 1], 700, 9, False),
    ([400, 383, 512, 384], 512, 17, True), ([120, 128, 33, 0, 97] * 4, 128, 7, True), ([300, 700, -1, 699, 129, 0, 1], 700, 9, True),
    ([64, 65, 128, 31, 32, 33, 500, 7] * 8, 520, 8, False), ([520] * 64, 520, 8, False), ([64, 65, 128, 31, 32, 257, 500, 7] * 8, 520, 8, True)])   # the last three: the roles as two launches
def test_places_of_the_backward(lens, L, H, causal):
    """The order in which the backward's workgroups are dealt, as its table has it."""
    B, tiles = len(lens), (L + 127) // 128
    S, (lut, radius) = 64, ops.delta_lut_device(32, 64, torch.device("cuda", 0))
    new = lambda *s: torch.zeros(*s, device="cuda", dtype=torch.bfloat16)
    x, tables = [new(B, L, H, 64) for _ in range(8)], [new(H, S, 64) for _ in range(4)]
    lse, length = torch.zeros(B * L, H, device="cuda"), torch.tensor(lens, dtype=torch.int32, device="cuda")
    a = _BwdArgs()
    for name, t in zip("q k v dout out dq dk dv pos_key pos_query d_pos_key d_pos_query lse seq_len delta_lut".split(), x + tables + [lse, length, lut]):
        setattr(a, name, t.data_ptr())
    for t in "q k v do out dq dk dv".split():
        for n, s in zip("bth", (L * H * 64, H * 64, 64)):
            setattr(a, f"{t}_stride_{n}", s)
    for t in "pk pq dp".split():
        setattr(a, t + "_stride_h", S * 64), setattr(a, t + "_stride_r", 64)
    a.batch, a.heads, a.head_dim, a.seqlen, a.att_span, a.lut_radius, a.dtype, a.causal, a.sm_scale = B, H, 64, L, S // 2, radius, _lib.FDB_BF16, causal, 0.1
    size = _lib.lib.fdb_attn_bwd_tables_workspace_bytes(ctypes.byref(a))
    seq_len, a.seq_len = a.seq_len, None
    assert size == _lib.lib.fdb_attn_bwd_tables_workspace_bytes(ctypes.byref(a))   # whoever asks does not have the lengths yet
    a.seq_len = seq_len
    ws = torch.full((size,), 0xFF, dtype=torch.uint8, device="cuda")
    a.workspace = ws.data_ptr()
    assert _lib.lib.fdb_attn_bwd_tables(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    n = B * tiles * H
    got = ws[size - (2 * n * 32 + 255) // 256 * 256:][:2 * n * 32].view(torch.int32).view(2 * n, 8).tolist()
    real = [min(max(l, 0), L) for l in lens]
    if 4 * sum(l < L - L // 4 for l in real) < B:
        dq, keys = [_plain_order(B, H, tiles, causal, k) for k in (False, True)]
        mixed = [("k", i) for i in range(n)] + [("q", i) for i in range(n)]
    else:
        dq, keys = [_order_by_length(real, H, tiles, causal, k) for k in (False, True)]
        mixed = [(r, i) for first in range(0, n, 32) for r in "kq" for i in range(first, min(n, first + 32))]
    if n > 2048:
        mixed = [("q", i) for i in range(n)] + [("k", i) for i in range(n)]
    want = [((keys if r == "k" else dq)[i], i, r == "k") for r, i in mixed]
    assert sorted(dq) == sorted(keys) == [(b, t, h) for b in range(B) for t in range(tiles) for h in range(H)]
    assert [((b, t, h), i, k == 1) for b, t, h, _, _, i, k, _ in got] == want
    assert [(first, tokens) for _, _, _, first, tokens, _, _, _ in got] == [(0, real[b]) for (b, _, _), _, _ in want]
