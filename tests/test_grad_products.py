"""The products of a layer's training backward (csrc/fdb_grad.hip) at the edges of their tiles, stages and shares, against the products in 64
bits; and the sizes they refuse."""
import ctypes

import pytest
import torch

from flashdeberta_amd import _lib

CODES = {torch.bfloat16: _lib.FDB_BF16, torch.float16: _lib.FDB_F16}


def _close(got, ref, scale, dtype, what):
    # one rounding of the result, and fp32 sums: 2^-22 of the sum of the terms' magnitudes covers the order of up to 2^12 additions that matter
    bound = torch.finfo(dtype).eps / 2 * ref.abs() * 1.01 + 2.0 ** -22 * scale + 1e-7
    assert ((got.double() - ref).abs() <= bound).all(), (what, ((got.double() - ref).abs() - bound).max().item())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("rows,depth,cols", [((1, 0), (64, 64), 64), ((0, 65), (64, 128), 128), ((64, 63), (192, 128), 192), ((200, 129), (320, 64), 448), ((1000, 512), (2304, 1536), 768),
                                             ((5500, 130), (64, 128), 768), ((9000, 65), (64, 192), 768),   # tiles of 128 rows: most compute units have one, most have two
                                             ((2700, 129), (128, 64), 768), ((2497, 0), (64, 64), 832)])   # tiles of 64 rows: a few compute units have two
def test_dgrad(rows, depth, cols, dtype):
    g = torch.Generator(device="cuda").manual_seed(sum(rows))
    w = torch.randn(max(depth), cols, device="cuda", generator=g).to(dtype)
    xs = [torch.randn(max(r, 1), d, device="cuda", generator=g).to(dtype) for r, d in zip(rows, depth)]
    outs = [torch.full((r + 1, cols), 7.0, device="cuda", dtype=dtype) for r in rows]
    p = lambda t, r: t.data_ptr() if r else None
    rc = _lib.lib.fdb_dgrad(p(xs[0], rows[0]), rows[0], depth[0], p(xs[1], rows[1]), rows[1], depth[1], w.data_ptr(), cols, p(outs[0], rows[0]), p(outs[1], rows[1]),
                            CODES[dtype], torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    for x, o, r, d in zip(xs, outs, rows, depth):
        assert (o[r:] == 7.0).all()
        if r:
            a, b = x.double(), w[:d].double()
            _close(o[:r], a @ b, a.abs() @ b.abs(), dtype, r)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,depth,cols", [((3000, 65), (64, 192), 768), ((2561, 0), (128, 64), 832), ((129, 4100), (448, 256), 640)])
def test_dgrad_of_one_round_of_tall_tiles(rows, depth, cols):
    """More tiles of 64 rows than compute units and no more of 128: fewer stages than the ring has, as many, and more."""
    test_dgrad(rows, depth, cols, torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("rows,x_cols,y_cols", [((1, 1), (192, 128), 64), ((63, 64), (384, 256), 128), ((65, 129), (320, 256), 192), ((200, 512), (576, 384), 256),
                                                ((1000, 512), (2304, 1536), 768), ((4096, 512), (2304, 1536), 768), ((700, 64), (192, 128), 1024)])
def test_wgrad(rows, x_cols, y_cols, dtype):
    g = torch.Generator(device="cuda").manual_seed(sum(rows) + y_cols)
    n = lambda r, c: torch.randn(r, c, device="cuda", generator=g).to(dtype)
    xs, ys = [n(r, c) for r, c in zip(rows, x_cols)], [n(r, y_cols) for r in rows]
    if rows[0] > 1:
        ys[0][-1, 0] = torch.inf   # the row that stages past the end re-read: it counts once, in its own column
    dw, db = torch.full((x_cols[0] + 1, y_cols), 7.0, device="cuda", dtype=dtype), torch.full((x_cols[0] + 8,), 7.0, device="cuda", dtype=dtype)
    ws = torch.empty(_lib.lib.fdb_wgrad_workspace_bytes(rows[0], rows[1], x_cols[0], y_cols), dtype=torch.uint8, device="cuda")
    got = []
    for _ in range(2):
        ws.fill_(0xFF)   # NaN: nothing of it is read before it is written
        rc = _lib.lib.fdb_wgrad(xs[0].data_ptr(), ys[0].data_ptr(), rows[0], x_cols[0], xs[1].data_ptr(), ys[1].data_ptr(), rows[1], x_cols[1], y_cols, dw.data_ptr(),
                                db.data_ptr(), ws.data_ptr(), CODES[dtype], torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        got.append((dw.clone(), db.clone()))
    assert (dw[x_cols[0]:] == 7.0).all() and (db[x_cols[0]:] == 7.0).all()
    assert all(torch.equal(a[:, 1:] if a.dim() == 2 else a, b[:, 1:] if b.dim() == 2 else b) for a, b in zip(*got))
    x0, x1, y0, y1 = [t.double() for t in (*xs, *ys)]
    ref, scale = x0.t() @ y0, x0.abs().t() @ y0.abs()
    ref[:x_cols[1]] += x1.t() @ y1
    scale[:x_cols[1]] += x1.abs().t() @ y1.abs()
    first = 1 if rows[0] > 1 else 0
    _close(dw[:x_cols[0], first:], ref[:, first:], scale[:, first:], dtype, "dw")
    if first:
        assert not dw[:x_cols[0], 0].isfinite().any()
    sums, scale = x0.sum(0), x0.abs().sum(0)
    sums[:x_cols[1]] += x1.sum(0)
    scale[:x_cols[1]] += x1.abs().sum(0)
    _close(db[:x_cols[0]], sums, scale, dtype, "db")


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(8, 8), (64, 64), (192, 344), (768, 768)])
def test_join(rows, cols):
    w = [torch.randn(rows, cols, device="cuda").to(torch.bfloat16) for _ in range(3)]
    b = [torch.randn(rows, device="cuda").to(torch.bfloat16) for _ in range(3)]
    out, bias = torch.full((3 * rows + 1, cols), 7.0, device="cuda", dtype=torch.bfloat16), torch.full((3 * rows + 8,), 7.0, device="cuda", dtype=torch.bfloat16)
    at = lambda ts: (ctypes.c_void_p * 3)(*[t.data_ptr() for t in ts])
    assert _lib.lib.fdb_join(at(w), at(b), out.data_ptr(), bias.data_ptr(), 2 * rows * cols, 2 * rows, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out[:-1], torch.cat(w)) and torch.equal(bias[:-8], torch.cat(b)) and (out[-1] == 7.0).all() and (bias[-8:] == 7.0).all()


def test_where_dgrad_serves():
    serves = _lib.lib.fdb_dgrad_serves
    assert serves(1, 0, 64) and serves(8192, 512, 768) and not serves(8192, 512, 1024) and serves(16384, 512, 768)


@pytest.mark.parametrize("change,code", [(dict(rows0=-1), -1), (dict(rows0=0, rows1=0), -5), (dict(cols=96), -5), (dict(depth1=96), -5), (dict(x0=24), -4), (dict(out1=0), -1), (dict(dtype=0), -2)])
def test_dgrad_refuses_on_the_host(change, code):
    kw = dict(x0=16, rows0=4, depth0=64, x1=32, rows1=4, depth1=64, w=48, cols=64, out0=64, out1=80, dtype=_lib.FDB_BF16)
    kw.update(change)
    assert _lib.lib.fdb_dgrad(*[v or None if k in ("x0", "x1", "w", "out0", "out1") else v for k, v in kw.items()], None) == code


@pytest.mark.parametrize("change,code", [(dict(rows1=0), -5), (dict(x_cols1=64), -5), (dict(x_cols1=256), -5), (dict(y_cols=72), -5), (dict(ws=48), -4), (dict(db=0), -1), (dict(dtype=3), -2)])
def test_wgrad_refuses_on_the_host(change, code):
    kw = dict(x0=16, y0=16, rows0=4, x_cols0=192, x1=32, y1=32, rows1=4, x_cols1=128, y_cols=64, dw=64, db=64, ws=96, dtype=_lib.FDB_BF16)
    kw.update(change)
    assert _lib.lib.fdb_wgrad(*[ctypes.c_void_p(v) if k in ("x0", "y0", "x1", "y1", "dw", "db", "ws") else v for k, v in kw.items()], None) == code
