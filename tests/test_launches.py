"""The launches that calls take (tests/launches.py: on the host, without a GPU)."""
import pytest

from flashdeberta_amd import _lib
from launches import P, launches


def _forward(batch, seqlen, heads=12, dtype=_lib.FDB_BF16, radius=512, workspace=0, **more):
    a = _lib.FdbAttnArgs()
    for n in ("q", "k", "v", "out", "pos_key", "pos_query", "lse", "delta_lut", "q_scale", "k_scale", "pk_scale", "pq_scale"):
        setattr(a, n, 0x1000)
    a.batch, a.heads, a.head_dim, a.dtype, a.max_seqlen, a.total_tokens = batch, heads, 64, dtype, seqlen, batch * seqlen
    a.att_span, a.lut_radius, a.sm_scale = radius // 2, radius, 0.1
    a.workspace, a.workspace_bytes = 0x100000 if workspace else None, workspace
    for n, v in more.items():
        setattr(a, n, v)
    return "fdb_attn_fwd", [a, None]


def _kinds(made):
    """far, near (the near steps alone), all (the near launch with the far tiles) or merge, and the shares"""
    out = []
    for name, _, shares, _ in made:
        all_tiles = "near" in name and name.split("EEv10FdbKParams")[0].endswith("Lb1E")
        out.append(("merge" if "merge" in name else "far" if "far8" in name or "attn_kernel" in name else "all" if all_tiles else "near", shares))
    return out


ALL = 1 << 32   # a workspace for whatever the call wants


@pytest.mark.parametrize("dtype", [_lib.FDB_BF16, _lib.FDB_F16, _lib.FDB_FP8_E4M3], ids=["bf16", "fp16", "e4m3"])
def test_where_the_near_launch_takes_the_far_tiles(dtype):
    """By the sizes alone: a caller without a workspace, whose tiles are not shared, takes the same kernels."""
    call = lambda *a, **kw: _forward(*a, dtype=dtype, **kw)
    cases = [
        (call(1, 575, workspace=ALL), [("near", 2), ("merge", 1)]),          # no key is far
        (call(1, 576, workspace=ALL), [("all", 2), ("merge", 1)]),
        (call(1, 576), [("all", 1)]),
        (call(1, 2048, 4, workspace=ALL), [("all", 4), ("merge", 1)]),
        (call(1, 2048, 4), [("all", 1)]),
        (call(64, 1152), [("all", 1)]),                                      # 8 far tiles at an end of the sequence
        (call(64, 1153), [("far", 1), ("near", 1)]),
        (call(2, 1152, 14), [("all", 1)]),
        (call(2, 1280, 12), [("all", 1)]),                                   # 240 query tiles on 256 compute units
        (call(2, 1300, 12), [("far", 1), ("near", 1)]),                      # 264
        (call(1, 2049), [("far", 1), ("near", 1)]),
        (call(8, 4096), [("far", 1), ("near", 1)]),
        (call(1, 960, radius=64), [("all", 1)]),                             # 12 far tiles at an end, 6 near ones in the middle
        (call(1, 961, radius=64), [("far", 1), ("near", 1)]),
        (call(1, 1000, causal=1), [("far", 1), ("near", 1)]),
        (call(1, 1000, far_splits=1), [("far", 1), ("near", 1)]),
        (call(1, 1000, near_splits=1), [("far", 1), ("near", 1)]),
        (call(1, 1000, cu_seqlens=0x1000, worklist=0x1000), [("far", 1), ("near", 1)]),
    ]
    for (_, want), (rc, made) in zip(cases, launches([c for c, _ in cases])):
        assert rc == 0 and _kinds(made) == want, (want, made)
    (_, whole), = launches([call(1, 1300)], cus=132)
    (_, short), = launches([call(1, 1300)], cus=131)
    assert _kinds(whole) == [("all", 1)] and _kinds(short)[0][0] == "far"


def _linear(rows, cols, depth, ldo=None, bias=P(0x1000)):
    return "fdb_linear", [P(0x1000), P(0x1000), bias, P(0x1000), rows, cols, depth, depth, depth, ldo or cols, _lib.FDB_BF16, None]


def test_an_error_of_the_runtime_ends_the_linear_layer():
    for rows in (24, 100):
        (rc, made), = launches([_linear(rows, 768, 768)], fails=1)
        assert rc == 719 and len(made) == 1, (rc, made)


def test_linear_layers_of_many_rows_are_tiled():
    """Columns or output rows by fours, a bias on any element, too: the streaming kernel reads all weights for every 32 rows.  It keeps what makes one
    workgroup a compute unit, and what the tiles are not built for."""
    calls = [_linear(200, 772, 768), _linear(200, 768, 768, ldo=772), _linear(200, 768, 768, bias=P(0x1002)), _linear(100, 768, 768), _linear(32, 772, 768),
             _linear(160, 772, 768), _linear(200, 770, 768), _linear(200, 768, 96)]
    for (rc, made), tiled in zip(launches(calls), [True] * 4 + [False] * 4):
        assert rc == 0 and len(made) == 1 and ("fdb_gemm_kernel" in made[0][0]) == tiled, made


def _gemm(rows, cols, depth, epilogue):
    return "fdb_gemm", [P(0x1000)] * 5 + [rows, cols, depth, depth, depth, cols, cols, epilogue, _lib.FDB_BF16, None]


def _dgrad(rows, cols):
    return "fdb_dgrad", [P(0x1000), rows, 3 * cols, P(0x1000), 0, 64, P(0x1000), cols, P(0x1000), P(0x1000), _lib.FDB_BF16, None]


def test_thresholds_of_the_products_follow_the_compute_units():
    """A device of half the compute units takes the kernels for half the rows, and serves it where this one serves twice as many."""
    rows = [256, 512, 1024, 1536, 2048, 3072, 4096, 8192, 16384]
    sizes = [(r, c, d, e) for r in rows for c in (768, 2304, 3072) for d in (768, 3072) for e in (0, 2)]
    asked = lambda part: ([_gemm(r // part, c, d, e) for r, c, d, e in sizes] + [_dgrad(r // part, c) for r in rows for c in (768, 1024)]
                          + [("fdb_gemm_serves", [r // part, c, d, e]) for r, c, d, e in sizes] + [("fdb_gemm_real_serves", [8 // part, r // 8, c, d, d]) for r, c, d, e in sizes]
                          + [("fdb_dgrad_serves", [r // part, 0, c]) for r in rows for c in (768, 1024)])
    whole, half = launches(asked(1), cus=256), launches(asked(2), cus=128)
    kernels = lambda made: [name for name, *_ in made]
    for call, (rc, made), (rc_half, made_half) in zip(asked(1), whole, half):
        assert rc == rc_half and kernels(made) == kernels(made_half), (call, made, made_half)
    assert len({k for _, made in whole for k in kernels(made)}) > 10   # every tile is among them


def test_where_near_workgroups_are_two_teams():
    """Where each has a compute unit to itself and ten steps or more; two shares that do not have one each become one of two teams."""
    cases = [(_forward(1, 288), 256, 1), (_forward(1, 289), 512, 1), (_forward(1, 128, 12), 256, 1), (_forward(3, 777), 512, 1), (_forward(4, 777), 256, 1),
             (_forward(1, 1024, workspace=ALL), 512, 2), (_forward(1, 2048, workspace=ALL), 512, 1), (_forward(1, 2048, 4, workspace=ALL), 512, 4),
             (_forward(1, 512, workspace=ALL), 256, 2), (_forward(1, 1536, workspace=ALL), 256, 3), (_forward(1, 1300, workspace=ALL), 256, 2),
             (_forward(2, 1024, workspace=ALL, causal=1), 512, 1), (_forward(3, 777, dtype=_lib.FDB_FP8_E4M3), 256, 1)]
    for (_, threads, shares), (rc, made) in zip(cases, launches([c for c, _, _ in cases])):
        near = [m for m in made if "near" in m[0]]
        assert rc == 0 and [m[2:] for m in near] == [(shares, threads)], (made, threads, shares)


@pytest.mark.parametrize("dtype", [_lib.FDB_BF16, _lib.FDB_F16, _lib.FDB_FP8_E4M3], ids=["bf16", "fp16", "e4m3"])
def test_the_workspace_asked_for_is_what_the_launches_use(dtype):
    """A slot for every far share but the first, and for every near share where there are two or more."""
    sizes = [(b, l, h, r) for b in (1, 2, 3, 5) for l in (100, 300, 512, 777, 1024, 1152, 1280, 1536, 1792, 2048, 3000, 4096) for h in (1, 4, 8, 12, 16) for r in (64, 512)]
    calls = [_forward(b, l, h, dtype, r, workspace=ALL, **more) for b, l, h, r in sizes for more in ({}, dict(causal=1), dict(near_splits=2), dict(cu_seqlens=0x1000, worklist=0x1000))]
    asked = launches([("fdb_attn_workspace_bytes", [args[0]]) for _, args in calls])
    slots = set()
    for (_, (a, _)), (want, _), (rc, made) in zip(calls, asked, launches(calls)):
        far, near = [max([shares for kind, shares in _kinds(made) if kind in kinds], default=1) for kinds in (("far",), ("near", "all"))]
        used = far - 1 + (near if near > 1 else 0)
        assert rc == 0 and want == used * a.total_tokens * a.heads * (64 * 2 + 4), (a.batch, a.max_seqlen, a.heads, a.lut_radius, made, want)
        slots.add(used)
    assert len(slots) > 4


def test_a_workspace_of_two_slots_where_three_shares_are_wanted():
    """One share of two teams, which two shares that crowd the compute units are slower than (1 x 1536 43.6 -> 40.8 us)."""
    two = 2 * 1536 * 12 * (64 * 2 + 4)
    (rc, made), = launches([_forward(1, 1536, workspace=two)])
    assert rc == 0 and [m[2:] for m in made] == [(1, 512)], made
