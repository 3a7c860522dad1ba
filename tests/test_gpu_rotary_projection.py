"""GPU parity of grl_rotary_attention: the projection whose epilogue rotates queries and keys (128 x 128 tiles on four and eight waves,
256 x 256 tiles, ragged last tiles, tiles whose slabs the waves share out) and the products that leave the rotation to attention, on rectangular and ragged batches, against the
float64 oracle of projection, rotation and attention on whole sequences.  Tolerances: max|y-ref|/max|ref| <= 1e-4 (fp32), 2e-2 (bf16)."""
import ctypes

import numpy as np
import pytest

from conftest import TOL_F32, TOL_BF16
from oracle import oracle_np as O
from grilly_amd import _lib as L

pytestmark = pytest.mark.gpu


# rows at 768 columns in bf16: 100 -> kernel 9, 400 -> 10, 810 -> 7 in the range of 8, 1500 -> 6, 3000 -> 4, 5390 -> 3; fp32: 27 and 100 -> kernel 9
# with the fp32 instruction, 300 -> with split operands; other head dims and more rows in fp32 rotate in attention
@pytest.mark.parametrize("dtype,B,S,H,D", [("bf16", 2, 50, 12, 64), ("bf16", 1, 7, 10, 64), ("bf16", 5, 80, 12, 64), ("bf16", 9, 90, 12, 64), ("bf16", 15, 100, 12, 64), ("bf16", 30, 100, 12, 64), ("bf16", 55, 98, 12, 64),
                                           ("bf16", 30, 100, 6, 128), ("bf16", 30, 100, 12, 32), ("bf16", 3, 700, 10, 64), ("fp32", 30, 100, 6, 64), ("fp32", 3, 9, 12, 64), ("fp32", 2, 50, 12, 64), ("fp32", 3, 100, 12, 64)])
@pytest.mark.parametrize("ragged", [False, True])
def test_rotary_attention(backend, dtype, B, S, H, D, ragged):
    c, code, d = backend.core, (L.GRL_BF16 if dtype == "bf16" else L.GRL_F32), H * D
    rng = np.random.default_rng(B + S + D)
    q = (lambda a: O.bf16_round(a)) if dtype == "bf16" else (lambda a: a)
    n = rng.integers(1, S + 1, B) if ragged else np.full(B, S)
    n[0] = S
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    M = int(off[-1])
    x = q(rng.standard_normal((M, d), dtype=np.float32))
    w = q((rng.standard_normal((3 * d, d)) / np.sqrt(d)).astype(np.float32))
    b = rng.standard_normal(3 * d).astype(np.float32)
    dx, dw, db = c.upload(x, code), c.upload(w, code), c.upload(b)
    do, dp = c.upload_raw(off), c.upload_raw(np.concatenate([np.arange(k) for k in n]).astype(np.int32))
    guard = np.full(M * d + 64, 7.0, np.float32)
    qkv, out = c.alloc(M * 3 * d * 4), c.upload(guard, code)
    try:
        if dtype == "fp32":          # one sequence with an infinity: the others stay what they are
            x[0, 1] = np.inf
            c.lib.grl_h2d(c.ctx, dx.ptr, x.ctypes.data, x.nbytes)
        rg = L.Ragged(do.ptr, dp.ptr, B, M, S)
        L.check(c.lib.grl_rotary_attention(c.ctx, code, B, S, ctypes.byref(rg) if ragged else None, H, D, dx.ptr, dw.ptr, db.ptr, None, qkv.ptr, out.ptr,
                                           10000.0, 1.0), "rotary_attention")
        got = c.download(out, (M * d + 64,), code)
        assert (got[M * d:] == 7.0).all() and np.isfinite(got[n[0] * d if dtype == "fp32" else 0:]).all()
        got = got[:M * d].reshape(M, H, D)
        for s in sorted({0, 1 % B, B // 2, B - 1} - ({0} if dtype == "fp32" else set())):
            rows = slice(off[s], off[s + 1])
            parts = O.truth_linear(x[rows], w, b).reshape(n[s], 3, H, D)
            ref = O.truth_attention(parts[None, :, 0], parts[None, :, 1], parts[None, :, 2], rope="half")
            assert O.max_rel(got[None, rows], ref) < (TOL_F32 if dtype == "fp32" else TOL_BF16), (s, n[s])
    finally:
        for t in (dx, dw, db, do, dp, qkv, out):
            t.free()


# (rows, head dim): products that rotate on tiles of 32 (100), 128 on eight waves (1500) and four (3000), 256 (5400); at head dim 32 a pass over the keys
@pytest.mark.parametrize("dtype,n,D", [("bf16", 50, 64), ("bf16", 750, 64), ("bf16", 1500, 64), ("bf16", 2700, 64), ("fp32", 50, 64), ("bf16", 50, 32)])
def test_positions_behind_the_table(backend, dtype, n, D):
    """Rows have to stand at positions 0, 1, 2 ...; others read nothing behind the table, whose last position (a power of two, 1024 at least) they take."""
    c, code, H = backend.core, (L.GRL_BF16 if dtype == "bf16" else L.GRL_F32), 12 * 64 // D
    base = 9000.0 + n + D + 7 * code          # a table of its own, no longer than it has to be
    d, M, end = H * D, 2 * n, max(1024, 1 << (n - 1).bit_length())
    rng = np.random.default_rng(n)
    bufs = dx, dw, db, do = [c.upload(rng.standard_normal((M, d), dtype=np.float32), code), c.upload((rng.standard_normal((3 * d, d)) / 30).astype(np.float32), code),
                             c.upload(rng.standard_normal(3 * d).astype(np.float32)), c.upload_raw(np.array([0, n, M], np.int32))]
    pos = np.concatenate([np.arange(n), np.arange(n) * 3 + end - n]).astype(np.int32)
    pos[-1] = 2 ** 31 - 1
    qkv, out = c.alloc(M * 3 * d * 4), c.alloc(M * d * 4)
    got = []
    for p in (np.minimum(pos, end - 1), pos):
        dp = c.upload_raw(p)
        L.check(c.lib.grl_rotary_attention(c.ctx, code, 0, 0, ctypes.byref(L.Ragged(do.ptr, dp.ptr, 2, M, n)), H, D, dx.ptr, dw.ptr, db.ptr, None, qkv.ptr, out.ptr,
                                           base, 1.0), "rotary_attention")
        got.append(c.download(out, (M, d), code))
        dp.free()
    np.testing.assert_array_equal(got[0], got[1])
    for t in bufs + [qkv, out]:
        t.free()


def test_no_table_where_nothing_reads_one(backend):
    """fp32 products of many rows leave the rotation to kernels that form their angles themselves (ragged batches)"""
    c, B, S, H, D = backend.core, 30, 100, 6, 64
    d, M = H * D, 3000
    bufs = dx, dw, do, dp, qkv, out = [c.alloc(M * d * 4), c.alloc(3 * d * d * 4), c.upload_raw(np.arange(0, M + 1, S, dtype=np.int32)),
                                       c.upload_raw(np.tile(np.arange(S, dtype=np.int32), B)), c.alloc(M * 3 * d * 4), c.alloc(M * d * 4)]
    for t in (dx, dw):
        L.check(c.lib.grl_memset(c.ctx, t.ptr, 0, t.nbytes), "memset")
    def in_use():
        stats = L.PoolStats()
        L.check(c.lib.grl_pool_get_stats(c.ctx, ctypes.byref(stats)), "pool")
        return stats.bytes_in_use
    before = in_use()
    L.check(c.lib.grl_rotary_attention(c.ctx, L.GRL_F32, B, S, ctypes.byref(L.Ragged(do.ptr, dp.ptr, B, M, S)), H, D, dx.ptr, dw.ptr, None, None, qkv.ptr, out.ptr,
                                       9998.0, 1.0), "rotary_attention")
    assert in_use() == before
    for t in bufs:
        t.free()


@pytest.mark.parametrize("dtype,B,S,D", [("bf16", 2, 50, 64), ("bf16", 15, 100, 64), ("bf16", 55, 98, 64), ("bf16", 5, 80, 32), ("fp32", 2, 50, 64), ("fp32", 30, 100, 64)])
def test_key_mask(backend, dtype, B, S, D):
    c, code, H = backend.core, (L.GRL_BF16 if dtype == "bf16" else L.GRL_F32), 12 * 64 // D
    d, M = H * D, B * S
    rng = np.random.default_rng(B * S)
    q = (lambda a: O.bf16_round(a)) if dtype == "bf16" else (lambda a: a)
    x, w, b = q(rng.standard_normal((M, d), dtype=np.float32)), q((rng.standard_normal((3 * d, d)) / np.sqrt(d)).astype(np.float32)), rng.standard_normal(3 * d).astype(np.float32)
    mask = (rng.random((B, S)) < 0.7).astype(np.float32)
    mask[-1] = np.arange(S) >= S // 2          # padding on the left
    mask[:, -1] = 1.0
    bufs = dx, dw, db, dm, qkv, out = [c.upload(x, code), c.upload(w, code), c.upload(b), c.upload(mask), c.alloc(M * 3 * d * 4), c.alloc(M * d * 4)]
    L.check(c.lib.grl_rotary_attention(c.ctx, code, B, S, None, H, D, dx.ptr, dw.ptr, db.ptr, dm.ptr, qkv.ptr, out.ptr, 10000.0, 1.0), "rotary_attention")
    got = c.download(out, (B, S, H, D), code)
    for s in sorted({0, B // 2, B - 1}):
        parts = O.truth_linear(x[s * S:(s + 1) * S], w, b).reshape(S, 3, H, D)
        ref = O.truth_attention(parts[None, :, 0], parts[None, :, 1], parts[None, :, 2], mask=mask[s:s + 1], rope="half")
        assert O.max_rel(got[s:s + 1], ref) < (TOL_F32 if dtype == "fp32" else TOL_BF16)
    for t in bufs:
        t.free()


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
def test_a_table_first_needed_under_capture(backend, dtype):
    """The launch that fills the cos/sin table is only recorded then: calls in front of the first replay do not use that table."""
    c, code, B, S, H, D = backend.core, (L.GRL_BF16 if dtype == "bf16" else L.GRL_F32), 2, 50, 12, 64
    d, M, base = H * D, B * S, 7001.0 + 8 * code                  # a base that nothing else uses
    rng = np.random.default_rng(6)
    q = (lambda a: O.bf16_round(a)) if dtype == "bf16" else (lambda a: a)
    x, w, b = q(rng.standard_normal((M, d), dtype=np.float32)), q((rng.standard_normal((3 * d, d)) / np.sqrt(d)).astype(np.float32)), rng.standard_normal(3 * d).astype(np.float32)
    bufs = dx, dw, db, do, dp, qkv, out = [c.upload(x, code), c.upload(w, code), c.upload(b), c.upload_raw(np.arange(0, M + 1, S, dtype=np.int32)),
                                           c.upload_raw(np.tile(np.arange(S, dtype=np.int32), B)), c.alloc(M * 3 * d * 4), c.alloc(M * d * 4)]
    rg = L.Ragged(do.ptr, dp.ptr, B, M, S)
    run = lambda: c.lib.grl_rotary_attention(c.ctx, code, 0, 0, ctypes.byref(rg), H, D, dx.ptr, dw.ptr, db.ptr, None, qkv.ptr, out.ptr, base, 1.0)
    parts = O.truth_linear(x, w, b).reshape(B, S, 3, H, D)
    ref = O.truth_attention(parts[:, :, 0], parts[:, :, 1], parts[:, :, 2], rope="half", base=base)
    stream, graph, replay = ctypes.c_void_p(c.lib.grl_stream(c.ctx)), ctypes.c_void_p(), ctypes.c_void_p()
    hip = lambda name, *args: L.check(getattr(c.lib, name)(*args), name)
    try:
        hip("hipStreamBeginCapture", stream, 2)          # relaxed: the table's allocation goes through
        rc = run()
        hip("hipStreamEndCapture", stream, ctypes.byref(graph))
        L.check(rc, "rotary_attention")
        hip("hipGraphInstantiate", ctypes.byref(replay), graph, None, None, ctypes.c_size_t(0))
        for _ in range(3):
            for launch in (lambda: L.check(run(), "rotary_attention"), lambda: hip("hipGraphLaunch", replay, stream)):
                L.check(c.lib.grl_memset(c.ctx, out.ptr, 0, out.nbytes), "memset")
                launch()
                assert O.max_rel(c.download(out, (B, S, H, D), code), ref) < (TOL_F32 if dtype == "fp32" else TOL_BF16)
    finally:
        if replay:
            c.lib.hipGraphExecDestroy(replay)
        if graph:
            c.lib.hipGraphDestroy(graph)
        for t in bufs:
            t.free()


def test_captures_share_one_table(backend):
    """Each capture records the filling once, into the same memory, and a call outside fills it again; all replays and calls agree."""
    c, code, B, S, H, D = backend.core, L.GRL_BF16, 2, 50, 12, 64
    d, M, base = H * D, B * S, 7103.0                            # a base that nothing else uses
    rng = np.random.default_rng(7)
    bufs = dx, dw, do, dp, qkv, out = [c.upload(rng.standard_normal((M, d), dtype=np.float32), code), c.upload((rng.standard_normal((3 * d, d)) / 28).astype(np.float32), code),
                                       c.upload_raw(np.arange(0, M + 1, S, dtype=np.int32)), c.upload_raw(np.tile(np.arange(S, dtype=np.int32), B)),
                                       c.alloc(M * 3 * d * 2), c.alloc(M * d * 2)]
    rg = L.Ragged(do.ptr, dp.ptr, B, M, S)
    run = lambda: L.check(c.lib.grl_rotary_attention(c.ctx, code, 0, 0, ctypes.byref(rg), H, D, dx.ptr, dw.ptr, None, None, qkv.ptr, out.ptr, base, 1.0), "rotary_attention")
    stream, graphs, replays = ctypes.c_void_p(c.lib.grl_stream(c.ctx)), [], []
    hip = lambda name, *args: L.check(getattr(c.lib, name)(*args), name)

    def in_use():
        stats = L.PoolStats()
        L.check(c.lib.grl_pool_get_stats(c.ctx, ctypes.byref(stats)), "pool")
        return stats.bytes_in_use

    def nodes(graph):
        n = ctypes.c_size_t()
        hip("hipGraphGetNodes", graph, None, ctypes.byref(n))
        return n.value
    try:
        before = in_use()
        for calls in (3, 1):
            graph, replay = ctypes.c_void_p(), ctypes.c_void_p()
            hip("hipStreamBeginCapture", stream, 2)              # relaxed: the table's allocation goes through
            try:
                for _ in range(calls):
                    run()
            finally:
                hip("hipStreamEndCapture", stream, ctypes.byref(graph))
            graphs.append(graph)
            hip("hipGraphInstantiate", ctypes.byref(replay), graph, None, None, ctypes.c_size_t(0))
            replays.append(replay)
        assert in_use() - before == 1024 * (D // 2) * 8
        assert (nodes(graphs[0]) - 1) == 3 * (nodes(graphs[1]) - 1)
        got = []
        for launch in [lambda r=r: hip("hipGraphLaunch", r, stream) for r in reversed(replays)] + [run] + [lambda r=r: hip("hipGraphLaunch", r, stream) for r in replays]:
            L.check(c.lib.grl_memset(c.ctx, out.ptr, 0, out.nbytes), "memset")
            launch()
            got.append(c.download(out, (M, d), code))
        assert np.isfinite(got[0]).all() and np.abs(got[0]).max() > 0
        for g in got[1:]:
            np.testing.assert_array_equal(g, got[0])
        assert in_use() - before == 1024 * (D // 2) * 8
    finally:
        for r in replays:
            c.lib.hipGraphExecDestroy(r)
        for g in graphs:
            c.lib.hipGraphDestroy(g)
        for t in bufs:
            t.free()
