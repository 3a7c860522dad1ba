"""GPU parity of the fp32 GEMM kernels that multiply split operands on the bf16 matrix cores (x = h + m + l, six plane products):
accuracy against float64, and operands that the split does not survive (infinities, NaN, values that round to bf16 infinity, products
that overflow), which the kernels compute again with the fp32 instruction.  The shapes reach every kernel: 32 x 32 tiles with shared K,
64 x 64, 64 x 128, 128 x 128 tiles on four and on eight waves, those with shares of the K loop, and 256 x 256 tiles, with one stage, fewer stages than are fetched ahead, odd numbers of them,
ragged rows and columns."""
import ctypes

import numpy as np
import pytest

from grilly_amd import _lib as L
from oracle import oracle_np as O

pytestmark = pytest.mark.gpu

SHAPES = [(1500, 384, 384), (1499, 416, 388),                                                 # 32 x 32
          (1501, 32, 1148), (1500, 64, 1152), (1500, 96, 1152), (1500, 160, 1152), (1500, 384, 1152),   # 64 x 64
          (1500, 768, 2304), (1499, 96, 1800), (3001, 32, 1148), (3001, 160, 1152),           # 128 x 128, eight waves
          (1500, 3072, 768), (1499, 3040, 764), (449, 3072, 1148), (799, 2080, 1148),         # the same in shares of K, the last one shorter
          (449, 3072, 768), (2999, 2080, 388),                                                # 32 x 32, long K
          (2001, 768, 3068), (4001, 768, 1536),                                               # 64 x 128
          (3000, 32, 2304), (2999, 64, 2300), (3000, 96, 2304), (3000, 768, 2304),            # 128 x 128
          (16380, 32, 2044), (16384, 64, 2048), (6399, 96, 2300), (6400, 768, 2304)]          # 256 x 256


def run(backend, x, W, b, epi=L.EPI_NONE):
    c = backend.core
    (M, K), N = x.shape, W.shape[0]
    dx, dw, db, dy = bufs = [c.upload(x), c.upload(W), c.upload(b), c.alloc(M * N * 4)]
    try:
        L.check(c.lib.grl_gemm_nt(c.ctx, L.GRL_F32, L.GRL_F32, M, N, K, dx.ptr, dw.ptr, db.ptr, dy.ptr, epi), "gemm_nt")
        return c.download(dy, (M, N))
    finally:
        for t in bufs:
            t.free()


def rel(y, ref):
    return np.linalg.norm(y - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("positive", [False, True])
def test_error_against_float64(backend, M, K, N, positive):
    """Roundings of a sum of K products to 24 bits, six per sixteen products: a random walk of at most sqrt(6 K / 16) steps of half
    a unit in the last place (2^-25 to 2^-24 of the result's size) where the terms have either sign, and what the nine-product
    expansion leaves out (2^-24); of terms of one sign the partial sums are smaller than the result."""
    rng = np.random.default_rng(M + K + N)
    make = (lambda *s: rng.random(s)) if positive else (lambda *s: rng.standard_normal(s))
    x, W, b = make(M, K).astype(np.float32), (make(N, K) / np.sqrt(K)).astype(np.float32), make(N).astype(np.float32)
    ref = x.astype(np.float64) @ W.T.astype(np.float64) + b
    bound = 2.0 ** -24 * (1 + np.sqrt(6 * K / 16))
    y = run(backend, x, W, b)
    assert rel(y, ref) < bound
    assert rel(run(backend, x, W, b, L.EPI_RELU), np.maximum(ref, 0)) < 2 * bound


@pytest.mark.parametrize("M,K,N", [(1500, 384, 384), (1500, 160, 1152), (1499, 96, 1800), (1499, 3040, 764), (3000, 96, 2304), (6399, 96, 2300)])
def test_operands_that_do_not_split(backend, M, K, N):
    rng = np.random.default_rng(M)
    x, W, b = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (N, K), (N,)))
    W[W == 0] = 1.0
    big = np.finfo(np.float32).max
    x[3, 5] = np.inf                             # +-inf by the sign of the weight
    x[40, 7], x[40, 9] = -np.inf, np.nan
    x[M - 1, 0], x[M - 1, 1] = np.inf, -np.inf   # NaN where the two products have opposite signs
    x[77] = 0.0
    x[77, 3] = big                               # rounds to bf16 infinity; times a small weight it is an ordinary number
    W[:, 3] = np.where(np.abs(W[:, 3]) < 0.5, W[:, 3], 0.25).astype(np.float32)
    W[11, 2] = np.nan
    b[5] = np.inf
    y = run(backend, x, W, b)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = x.astype(np.float64) @ W.T.astype(np.float64) + b
        ref = np.where(np.abs(ref) > big, np.sign(ref) * np.inf, ref)
    ok = np.isfinite(ref)
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))
    np.testing.assert_array_equal(y[~ok & ~np.isnan(ref)], ref[~ok & ~np.isnan(ref)].astype(np.float32))
    assert np.allclose(y[77][ok[77]], ref[77][ok[77]], rtol=1e-5, atol=0)
    rows = np.ones(M, bool)
    rows[77] = False
    okr = ok[rows]
    assert rel(y[rows][okr], ref[rows][okr]) < 2.0 ** -24 * (1 + np.sqrt(K))


@pytest.mark.parametrize("M,K,N", [(33, 96, 100), (1500, 384, 384), (1501, 32, 1148), (1501, 160, 1148), (3001, 96, 1152), (6399, 96, 1148)])
def test_gated_error_against_float64(backend, M, K, N):
    """Both sums as above; an activation that adds no error of its own: g * relu(u)."""
    c, rng = backend.core, np.random.default_rng(M + K + N)
    x, (Wg, Wu), (bg, bu) = rng.standard_normal((M, K)).astype(np.float32), (rng.standard_normal((2, N, K)) / np.sqrt(K)).astype(np.float32), rng.standard_normal((2, N)).astype(np.float32)
    bufs = [c.upload(a) for a in (x, Wg, Wu, bg, bu)] + [c.alloc(M * N * 4)]
    try:
        L.check(c.lib.grl_glu_nt(c.ctx, L.GRL_F32, L.GRL_F32, M, N, K, *(t.ptr for t in bufs), None, None, L.EPI_RELU), "glu_nt")
        y = c.download(bufs[-1], (M, N))
    finally:
        for t in bufs:
            t.free()
    g, u = (x.astype(np.float64) @ w.T.astype(np.float64) + b for w, b in ((Wg, bg), (Wu, bu)))
    assert rel(y, g * np.maximum(u, 0)) < 3 * 2.0 ** -24 * (1 + np.sqrt(6 * K / 16))


def test_small_and_large_values(backend):
    """The planes of a float of any ordinary exponent are bf16 numbers: scaling by powers of two changes nothing."""
    rng = np.random.default_rng(5)
    x, W, b = (rng.standard_normal(s).astype(np.float32) for s in ((3000, 96), (2304, 96), (2304,)))
    y = run(backend, x, W, b)
    for e, f in ((-60, 30), (90, -40), (-20, -40)):
        s, t = np.float32(2.0 ** e), np.float32(2.0 ** f)
        np.testing.assert_array_equal(run(backend, x * s, W * t, b * (s * t)), y * (s * t))


# where the 32 x 32 tiles' four sums on the fp32 instruction were the fastest before the split operands, and more than one 128 x 128
# tile per CU all the same; plain and gated
FOUR_SUMS = [(2722, 3072, 2304, False), (8251, 3072, 768, False), (2722, 4096, 3072, False), (6400, 4096, 1024, False), (800, 2048, 8192, False),
             (800, 8192, 4096, True), (6400, 11008, 512, True)]


@pytest.mark.parametrize("M,K,N,gated", FOUR_SUMS)
def test_four_sums_where_four_were(backend, M, K, N, gated):
    """R = 6 K / 16 roundings walk along one sum whose size grows with the root of its length: an error of e sqrt(R / 2); along four sums of
    a quarter each it is e sqrt(R / 8), half of it.  Measured at K = 768: 4.2e-7 and 2.0e-7, i.e. 0.42 and 0.20 times 2^-24 sqrt(R).  The
    bound lies between the two."""
    rng = np.random.default_rng(M + K + N)
    x, W = rng.standard_normal((M, K)).astype(np.float32), (rng.standard_normal((2 if gated else 1, N, K)) / np.sqrt(K)).astype(np.float32)
    bound = 2.0 ** -24 * 0.29 * np.sqrt(6 * K / 16)
    rows = slice(0, 257)                          # (float64 in full would take a minute)
    ref = [x[rows].astype(np.float64) @ w.T.astype(np.float64) for w in W]
    if not gated:
        y = run(backend, x, W[0], np.zeros(N, np.float32))
        assert rel(y[rows], ref[0]) < bound
        return
    c = backend.core
    bufs = [c.upload(x), c.upload(W[0]), c.upload(W[1]), c.alloc(M * N * 4)]
    try:
        L.check(c.lib.grl_glu_nt(c.ctx, L.GRL_F32, L.GRL_F32, M, N, K, *(t.ptr for t in bufs[:3]), None, None, bufs[3].ptr, None, None, L.EPI_RELU), "glu_nt")
        y = c.download(bufs[3], (M, N))
    finally:
        for t in bufs:
            t.free()
    assert rel(y[rows], ref[0] * np.maximum(ref[1], 0)) < 1.5 * bound      # two independent sums: sqrt(2)


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_one_term(backend, M, K, N):
    """A sum of one product (a row selector, a diagonal scaling).  The largest of its six plane products comes last, so the sum is rounded
    at its own size once (measured: to within a unit in the last place, 2^-23), and what is left out is at most 2^-24: m and l are
    up to 2^-8 and 2^-17 of an operand.  Measured 1.5e-7; with the largest product third, 2.8e-7."""
    rng = np.random.default_rng(M + K + N)
    x, W = np.zeros((M, K), np.float32), rng.standard_normal((N, K)).astype(np.float32)
    at, val = rng.integers(0, K, M), rng.standard_normal(M).astype(np.float32)
    x[np.arange(M), at] = val
    y = run(backend, x, W, np.zeros(N, np.float32))
    ref = W.astype(np.float64).T[at] * val[:, None].astype(np.float64)
    assert (np.abs(y - ref) / np.maximum(np.abs(ref), 1e-30)).max() < 3 * 2.0 ** -24


@pytest.mark.parametrize("M,K,N", [(1500, 384, 384), (1499, 160, 1152), (1500, 768, 2304), (1499, 3040, 764), (2001, 768, 3068), (3000, 768, 2304), (3000, 768, 2303), (6400, 768, 2304)])
@pytest.mark.parametrize("ex,ew", [(-112, 100), (100, -112), (-120, 124), (-125, 60), (60, -125), (-118, 0), (0, -118), (-70, -45), (60, 40), (110, -120)])
def test_operands_far_below_one(backend, M, K, N, ex, ew):
    """Operands near the smallest normal number: every bit of theirs counts as it does elsewhere (the bound of test_error_against_float64).
    The last two overflow at the size that operands are split at and are formed with the fp32 instruction (one rounding per product)."""
    rng = np.random.default_rng(M + K + N)
    x, W = rng.standard_normal((M, K)).astype(np.float32) * np.float32(2.0 ** ex), (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32) * np.float32(2.0 ** ew)
    y = run(backend, x, W, np.zeros(N, np.float32)).astype(np.float64)
    rows = slice(0, 257)
    ref = x[rows].astype(np.float64) @ W.T.astype(np.float64)
    assert rel(y[rows], ref) < 2.0 ** -24 * (1 + np.sqrt(K if ex + ew >= 80 or ex > 104 else 6 * K / 16))


@pytest.mark.parametrize("M,K,N,dtype", [(1499, 3040, 764, "fp32"), (128, 3072, 768, "fp32"), (128, 4096, 768, "bf16"),      # 128 x 128 and 32 x 32 tiles
                                         (100, 1000, 256, "fp32"), (100, 2056, 256, "bf16")])                          # the register-staged 64 x 64 tiles
def test_shares_of_k_take_nothing_from_the_pool_under_capture(backend, M, K, N, dtype):
    """A captured graph would keep the address of the shares after the pool has given it away: a product that runs in shares of K
    otherwise is recorded without them, and its replays give what new inputs ask for."""
    c, rng = backend.core, np.random.default_rng(8)
    code, q = (L.GRL_BF16, lambda a: O.bf16_round(a.astype(np.float32))) if dtype == "bf16" else (L.GRL_F32, lambda a: a.astype(np.float32))
    W, b = q(rng.standard_normal((N, K)) / np.sqrt(K)), rng.standard_normal(N).astype(np.float32)
    inputs = [q(np.random.default_rng(seed).standard_normal((M, K))) for seed in range(3)]
    dx, dw, db, dy, *dxs = bufs = [c.upload(inputs[0], code), c.upload(W, code), c.upload(b), c.alloc(M * N * 4)] + [c.upload(x, code) for x in inputs]
    product = lambda x: c.lib.grl_gemm_nt(c.ctx, code, L.GRL_F32, M, N, K, x.ptr, dw.ptr, db.ptr, dy.ptr, L.EPI_NONE)
    stream, graph, run_it = ctypes.c_void_p(c.lib.grl_stream(c.ctx)), ctypes.c_void_p(), ctypes.c_void_p()
    hip = lambda name, *args: L.check(getattr(c.lib, name)(*args), name)
    try:
        before = c.pool_stats()
        hip("hipStreamBeginCapture", stream, 2)          # relaxed: an allocation would go through
        rc = product(dx)
        hip("hipStreamEndCapture", stream, ctypes.byref(graph))
        L.check(rc, "gemm_nt")
        assert c.pool_stats() == before
        hip("hipGraphInstantiate", ctypes.byref(run_it), graph, None, None, ctypes.c_size_t(0))
        for x, d in zip(inputs, dxs):
            hip("hipMemcpyAsync", ctypes.c_void_p(dx.ptr), ctypes.c_void_p(d.ptr), ctypes.c_size_t(x.size * (2 if dtype == "bf16" else 4)), 3, stream)
            hip("hipGraphLaunch", run_it, stream)
            ref = x.astype(np.float64) @ W.T.astype(np.float64) + b
            assert rel(c.download(dy, (M, N)), ref) < 2.0 ** -24 * (1 + np.sqrt(K))      # bf16 products are exact; up to K roundings
            L.check(product(dxs[0]), "gemm_nt")          # eager work between the replays takes and returns the pool's blocks
    finally:
        if run_it:
            c.lib.hipGraphExecDestroy(run_it)
        if graph:
            c.lib.hipGraphDestroy(graph)
        for t in bufs:
            t.free()


@pytest.mark.parametrize("M,K,N", [(300, 3072, 768), (351, 3072, 768), (639, 3072, 768), (449, 4096, 1024), (1201, 2048, 512), (1999, 1152, 764)])
def test_shares_in_place_of_two_small_tiles_a_unit(backend, M, K, N):
    """In shares of K where a compute unit would get two 32 x 32 tiles or more of a long K (the first size: one, no shares); under capture without."""
    rng = np.random.default_rng(M + K + N)
    x, W, b = rng.standard_normal((M, K)).astype(np.float32), (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    assert rel(run(backend, x, W, b), x.astype(np.float64) @ W.T.astype(np.float64) + b) < 2.0 ** -24 * (1 + np.sqrt(6 * K / 16))
    test_shares_of_k_take_nothing_from_the_pool_under_capture(backend, M, K, N, "fp32")


@pytest.mark.parametrize("M,K,N", [(1999, 1152, 764), (1688, 992, 764), (300, 3072, 768), (33, 2080, 388),      # one workgroup a tile: split operands, then the fp32 instruction
                                   (1753, 1152, 764), (1688, 1024, 764)])                                      # shares
@pytest.mark.parametrize("positive", [False, True])
def test_small_tiles_of_a_long_sum(backend, M, K, N, positive):
    """32 x 32 tiles (test_dispatch_host pins which of these sizes take them) and the shares that stand in for them, K of 31 slabs and more"""
    test_error_against_float64(backend, M, K, N, positive)


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("M,K,N", [(1499, 384, 1152), (3001, 384, 1152), (9793, 384, 1536), (9791, 64, 1528), (257, 128, 264)])
def test_every_element_of_the_staged_epilogues(backend, dtype, M, K, N):
    """Folded LayerNorm with GELU and the plain product with residual, every element against float64: each output chunk is a 16-byte
    buffer store whose registers are reused at once.  Rows and columns end inside tiles; what lies behind the matrix stays."""
    c, bf = backend.core, dtype == "bf16"
    code, pad = (L.GRL_BF16 if bf else L.GRL_F32), 64
    rng = np.random.default_rng(M + K + N)
    q = (lambda a: O.bf16_round(a.astype(np.float32))) if bf else (lambda a: a.astype(np.float32))
    x, W, r = q(rng.standard_normal((M, K))), q(rng.standard_normal((N, K)) / np.sqrt(K)), q(rng.standard_normal((M, N)))
    b, cs = rng.standard_normal(N).astype(np.float32), W.sum(1, dtype=np.float64).astype(np.float32)
    st = (rng.random((M, 2)) + 0.5).astype(np.float32)
    dx, dw, db, dc, ds, dr, dy = bufs = [c.upload(x, code), c.upload(W, code), c.upload(b), c.upload(cs), c.upload(st), c.upload(r, code),
                                         c.upload(np.full(M * N + pad, 7.0, np.float32), code)]
    acc = x.astype(np.float64) @ W.T.astype(np.float64)
    tol = 2e-2 if bf else 1e-5
    try:
        L.check(c.lib.grl_ln_gemm_nt_stats(c.ctx, code, code, M, N, K, dx.ptr, dw.ptr, dc.ptr, db.ptr, ds.ptr, dy.ptr, L.EPI_GELU), "ln_gemm_nt_stats")
        got = c.download(dy, (M * N + pad,), code)
        ref = O.truth_gelu(acc * st[:, :1] - st[:, 1:] * cs.astype(np.float64) + b)
        assert np.abs(got[:M * N].reshape(M, N) - ref).max() < tol * np.abs(ref).max() and (got[M * N:] == 7.0).all()
        L.check(c.lib.grl_gemm_nt_res(c.ctx, code, code, M, N, K, dx.ptr, dw.ptr, db.ptr, dr.ptr, dy.ptr), "gemm_nt_res")
        got = c.download(dy, (M * N + pad,), code)
        ref = acc + b + r
        assert np.abs(got[:M * N].reshape(M, N) - ref).max() < tol * np.abs(ref).max() and (got[M * N:] == 7.0).all()
    finally:
        for t in bufs:
            t.free()


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_layernormed_residual_with_rows_beyond_a_buffer_offset(backend, dtype):
    """Output rows of 8 MiB: 256 of them span 2 GiB, where the kernels address every chunk by itself."""
    c, bf = backend.core, dtype == "bf16"
    code, es, K, M = (L.GRL_BF16, 2, 64, 2) if bf else (L.GRL_F32, 4, 32, 2)
    reps = 4097 if bf else 2049
    N = 1024 * reps
    rng = np.random.default_rng(3)
    q = (lambda a: O.bf16_round(a.astype(np.float32))) if bf else (lambda a: a.astype(np.float32))
    A, Wb, Rb = q(rng.standard_normal((M, K))), q(rng.standard_normal((1024, K)) / np.sqrt(K)), q(rng.standard_normal((M, 1024)))
    g, b, bt = (rng.standard_normal(1024).astype(np.float32) for _ in range(3))
    st = np.array([[0.9, 0.1], [1.1, -0.2]], np.float32)
    ref = A.astype(np.float64) @ Wb.T.astype(np.float64) + b + (Rb.astype(np.float64) * st[:, :1] - st[:, 1:]) * g + bt
    bufs = [c.upload(np.tile(Wb, (reps, 1)), code), c.upload(A, code), c.upload(np.tile(b, reps)), c.upload(np.tile(Rb, (1, reps)), code), c.upload(st),
            c.upload(np.tile(g, reps)), c.upload(np.tile(bt, reps)), c.alloc(M * N * es), c.alloc(M * 8), c.alloc(c.lib.grl_gemm_nt_resln_workspace(M, N))]
    dw, da, db, dr, ds, dg, dbt, dy, so, wk = bufs
    try:
        L.check(c.lib.grl_gemm_nt_resln(c.ctx, code, M, N, K, da.ptr, dw.ptr, db.ptr, dr.ptr, ds.ptr, dg.ptr, dbt.ptr, dy.ptr, 1e-5, so.ptr, wk.ptr), "resln")
        y = c.download(dy, (M, N), code).reshape(M, reps, 1024)
        assert np.abs(y - ref[:, None, :]).max() < (2e-2 if bf else 1e-5) * np.abs(ref).max()
        stats = c.download(so, (M, 2))
        sd = np.sqrt(ref.var(1) + 1e-5)
        assert np.allclose(stats[:, 0], 1 / sd, rtol=5e-3 if bf else 1e-4) and np.allclose(stats[:, 1], ref.mean(1) / sd, atol=5e-3 if bf else 1e-4)
    finally:
        for t in bufs:
            t.free()
