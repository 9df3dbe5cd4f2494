"""Products with what follows them (csrc/fdb_gemm.hip): each tile shape at its remainders, against the product in 64 bits, and GELU at
the values its table leaves out."""
import pytest
import torch
import torch.nn.functional as F

from flashdeberta_amd import _lib

PLAIN, GELU, RESIDUAL = 0, 1, 2


def _run(x, w, bias, epilogue, residual=None):
    M, N = x.shape[0], w.shape[0]
    out = torch.full((M + 1, N + 8), 7.0, device=x.device, dtype=x.dtype)   # a stride of its own, and what must not be written
    code = {torch.bfloat16: _lib.FDB_BF16, torch.float16: _lib.FDB_F16}[x.dtype]
    rc = _lib.lib.fdb_gemm(x.data_ptr(), w.data_ptr(), None if bias is None else bias.data_ptr(), None if residual is None else residual.data_ptr(), out.data_ptr(),
                           M, N, x.shape[1], x.stride(0), w.stride(0), out.stride(0), 0 if residual is None else residual.stride(0), epilogue, code,
                           torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert (out[M] == 7.0).all() and (out[:, N:] == 7.0).all()
    return out[:M, :N]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("M,N,K", [
    (1, 8, 64), (33, 72, 128), (100, 136, 320),      # 32 x 64, contractions shorter and longer than the stages under way
    (1030, 520, 64), (1030, 520, 256),               # 64 x 64
    (1601, 1360, 64), (1601, 1360, 320),             # 64 x 192, four stages
    (3000, 1160, 64), (3000, 1160, 192),             # 64 x 192, two workgroups a compute unit
    (5000, 1400, 64), (5000, 1400, 128),             # 256 x 192
])
def test_tiles_and_their_remainders(M, N, K, dtype):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w = [(torch.randn(r, K + 8, device="cuda", generator=g) * s).to(dtype)[:, :K] for r, s in ((M, 1.0), (N, K ** -0.5))]
    bias, residual = torch.randn(N, device="cuda", generator=g).to(dtype), torch.randn(M, N + 8, device="cuda", generator=g).to(dtype)[:, :N]
    y = x.double() @ w.double().t()
    eps = torch.finfo(dtype).eps / 2   # the largest relative error of one rounding; the fp32 sums' own is smaller by 2^-10
    for epilogue, b, ref, roundings in ((PLAIN, None, y, 1), (PLAIN, bias, y + bias.double(), 1), (GELU, bias, F.gelu(y + bias.double()), 2),
                                        (RESIDUAL, bias, y + bias.double() + residual.double(), 2)):
        got = _run(x, w, b, epilogue, residual if epilogue == RESIDUAL else None).double()
        # a rounding of y moves gelu(y) by at most 1.13 times as much, and y + residual by |y|'s rounding
        bound = eps * (ref.abs() + (roundings - 1) * 1.13 * (y + bias.double()).abs()) * 1.01 + 1e-5
        assert ((got - ref).abs() <= bound).all(), (epilogue, ((got - ref).abs() - bound).max().item())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1030, 1160, 64), (1030, 1160, 256), (961, 1032, 192)])
def test_tiles_of_64_by_four_waves(M, N, K):
    """More tiles of 64 x 64 than compute units, up to where wider ones begin; (1030, 520) is eight waves'."""
    test_tiles_and_their_remainders(M, N, K, torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("M,N,K", [(33, 4, 64), (200, 772, 128), (1030, 516, 64), (1601, 1364, 64), (3000, 1164, 64), (5000, 1404, 64)])   # streamed, then each tile
@pytest.mark.parametrize("pitch,shift", [(0, 0), (4, 0), (0, 1), (4, 3), (8, 2)])   # of the output's rows beyond N, and elements the bias is off 8 bytes by
def test_linear_by_fours(M, N, K, pitch, shift, dtype):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w = [(torch.randn(r, K, device="cuda", generator=g) * s).to(dtype) for r, s in ((M, 1.0), (N, K ** -0.5))]
    bias = torch.randn(N + shift, device="cuda", generator=g).to(dtype)[shift:]
    out = torch.full((M + 1, N + pitch), 7.0, device="cuda", dtype=dtype)
    assert _lib.lib.fdb_linear(x.data_ptr(), w.data_ptr(), bias.data_ptr(), out.data_ptr(), M, N, K, K, K, N + pitch,
                               {torch.bfloat16: _lib.FDB_BF16, torch.float16: _lib.FDB_F16}[dtype], torch.cuda.current_stream().cuda_stream) == 0
    assert (out[M] == 7.0).all() and (out[:, N:] == 7.0).all()
    ref = x.double() @ w.double().t() + bias.double()
    bound = torch.finfo(dtype).eps / 2 * ref.abs() * 1.01 + 1e-5   # one rounding of the result; the fp32 sums' own is smaller by 2^-10
    assert ((out[:M, :N].double() - ref).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_gelu_of_every_value_is_torchs(dtype):
    """The product of zeros leaves the bias: all 65536 patterns, in rows of their own and beside ordinary values."""
    every = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(dtype)
    for values in (every, torch.where(torch.arange(65536, device="cuda") % 64 == 5, every, torch.ones_like(every))):
        x, w = torch.zeros(3, 64, device="cuda", dtype=dtype), torch.zeros(65536, 64, device="cuda", dtype=dtype)
        got, ref = _run(x, w, values, GELU), F.gelu(values + 0)
        assert torch.equal(got[0].isnan(), ref.isnan()) and torch.equal(got.nan_to_num(), ref.nan_to_num().expand(3, -1))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("kinds", ["tiny ordinary", "ordinary large", "zero tiny large", "zero tiny ordinary large", "denormal tiny large", "ordinary large inf", "tiny ordinary nan"])
def test_gelu_of_unlike_values_side_by_side(kinds, dtype):
    """Of the values a wave looks at together some are in the table, some halves, some themselves or nothing, some neither: each row another mixture."""
    every = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(dtype)
    size, least = every.float().abs(), torch.finfo(dtype).tiny
    of = {"zero": size == 0, "denormal": (size > 0) & (size < least), "tiny": (size >= least) & (size < 2.0 ** -14 + least), "ordinary": (size > 2.0 ** -14) & (size < 8),
          "large": (size >= 8) & size.isfinite(), "inf": size.isinf(), "nan": size.isnan()}
    g = torch.Generator(device="cuda").manual_seed(len(kinds))
    pick = lambda some, n: some[torch.randint(len(some), (n,), device="cuda", generator=g)]
    rows = torch.stack([pick(every[of[k]], 8192) for k in kinds.split()])
    mixed = rows.gather(0, torch.randint(len(rows), (70, 8192), device="cuda", generator=g))
    if set(kinds.split()) & {"denormal", "inf", "nan"}:   # as the bias, alike in all rows: 0 x inf is none of them
        x, w, bias = torch.zeros(70, 128, device="cuda", dtype=dtype), torch.zeros(8192, 128, device="cuda", dtype=dtype), mixed[0].contiguous()
        mixed = bias.expand(70, -1)
    else:                                                 # y = x . w^T to the bit: x the identity, the columns of w the rows of y
        x, w, bias = torch.eye(70, 128, device="cuda", dtype=dtype), torch.zeros(8192, 128, device="cuda", dtype=dtype), None
        w[:, :70] = mixed.t()
    got, ref = _run(x, w, bias, GELU), F.gelu(mixed + 0)   # (-0 + 0 is 0, as in the sums)
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.nan_to_num(), ref.nan_to_num())


def test_where_it_serves():
    serves = _lib.lib.fdb_gemm_serves
    assert not serves(32, 768, 768, RESIDUAL) and serves(33, 768, 768, RESIDUAL) and not serves(64, 768, 100, RESIDUAL) and not serves(64, 772, 768, GELU)
    assert not serves(64, 768, 3072, RESIDUAL) and serves(4096, 768, 3072, RESIDUAL)      # few tiles and a long contraction
    assert serves(2048, 2304, 768, PLAIN) and not serves(4096, 2304, 768, PLAIN)


@pytest.mark.parametrize("change,code", [(dict(rows=0), "SHAPE"), (dict(cols=12), "SHAPE"), (dict(depth=96), "SHAPE"), (dict(ldx=56), "SHAPE"), (dict(ldx=(1 << 22) + 8), "SHAPE"),
                                         (dict(x=24), "ALIGN"), (dict(bias=20), "ALIGN"), (dict(ldo=68), "ALIGN"), (dict(residual=0), "NULL"), (dict(residual=8), "ALIGN"),
                                         (dict(ldr=56), "SHAPE"), (dict(dtype=0), "DTYPE"), (dict(epilogue=3), "UNSUPPORTED")])
def test_refused_on_the_host(change, code):
    codes = {"NULL": -1, "DTYPE": -2, "ALIGN": -4, "SHAPE": -5, "UNSUPPORTED": -10}
    kw = dict(x=16, w=32, bias=48, residual=64, out=80, rows=64, cols=64, depth=64, ldx=64, ldw=64, ldo=64, ldr=64, epilogue=RESIDUAL, dtype=_lib.FDB_BF16)
    kw.update(change)
    rc = _lib.lib.fdb_gemm(*[v or None if k in ("x", "w", "bias", "residual", "out") else v for k, v in kw.items()], None)
    assert rc == codes[code], (rc, code)
