"""GPU parity of the bf16 256 x 256 kernel whose K steps run in phases: two workgroup tiles in a row and a ragged last row and column
tile, with the fewest steps it takes, odd and even step counts (the LDS stage a tile starts in alternates), against float64 sums.
Tolerance: max|y-ref|/max|ref| <= 2e-2, as in the other bf16 GEMM tests."""
import numpy as np
import pytest

import test_gpu_ln_linear as lnl
from conftest import TOL_BF16
from oracle import oracle_np as O
from grilly_amd import _lib as L

pytestmark = pytest.mark.gpu

M, N = 64 * 256 - 37, 8 * 256 - 8          # 512 tiles: two for each compute unit


def rows_of(rng):
    edges = np.concatenate([np.arange(0, M, 256), np.minimum(np.arange(255, M + 256, 256), M - 1)])
    return np.unique(np.concatenate([edges, rng.integers(0, M, 100)]))


@pytest.mark.parametrize("slabs", [2, 3, 4, 7])
@pytest.mark.parametrize("kind", ["gelu", "residual", "folded", "gated", "f32_out", "odd_columns", "normed_residual"])
def test_phased_tiles(backend, kind, slabs):
    c, B, K = backend.core, L.GRL_BF16, 64 * slabs
    rng = np.random.default_rng(slabs)
    q = lambda a: O.bf16_round(a.astype(np.float32))
    n = N - 3 if kind == "odd_columns" else N // 2 if kind == "gated" else N
    x, w, b, r = q(rng.standard_normal((M, K), dtype=np.float32) + 0.5), q(rng.standard_normal((n, K)) / np.sqrt(K)), rng.standard_normal(n).astype(np.float32), rows_of(rng)
    res = q(rng.standard_normal((M, n), dtype=np.float32)) if "residual" in kind else np.zeros((1, n), np.float32)
    guard = np.full(M * n + 64, 7.0, np.float32)
    sums = w.astype(np.float64).sum(1).astype(np.float32)
    mean, sd = x.astype(np.float64).mean(1), x.astype(np.float64).std(1)
    stats = np.stack([1 / sd, mean / sd], 1).astype(np.float32)
    out = L.GRL_F32 if kind == "f32_out" else B
    dx, dw, db, dr, ds, dst, dy = bufs = [c.upload(x, B), c.upload(w, B), c.upload(b), c.upload(res, B), c.upload(sums), c.upload(stats), c.upload(guard, out)]
    try:
        pre = O.truth_linear(x[r], w, b)
        if kind == "gelu":
            L.check(c.lib.grl_gemm_nt(c.ctx, B, B, M, n, K, dx.ptr, dw.ptr, db.ptr, dy.ptr, L.EPI_GELU), "gemm_nt")
            ref = O.truth_gelu(pre)
        elif kind == "residual":
            L.check(c.lib.grl_gemm_nt_res(c.ctx, B, B, M, n, K, dx.ptr, dw.ptr, db.ptr, dr.ptr, dy.ptr), "gemm_nt_res")
            ref = pre + res[r].astype(np.float64)
        elif kind == "folded":
            L.check(c.lib.grl_ln_gemm_nt_stats(c.ctx, B, B, M, n, K, dx.ptr, dw.ptr, ds.ptr, db.ptr, dst.ptr, dy.ptr, L.EPI_NONE), "ln_gemm_nt_stats")
            ref = O.truth_linear((x[r] - mean[r, None]) / sd[r, None], w, b)
        elif kind == "normed_residual":
            eps, rst = 1e-5, np.stack([1 / res.astype(np.float64).std(1), res.astype(np.float64).mean(1) / res.astype(np.float64).std(1)], 1).astype(np.float32)
            dg, dbt, drs, dso, dws = c.upload(1 + b / 10), c.upload(sums / 10), c.upload(rst), c.alloc(M * 8), c.alloc(c.lib.grl_gemm_nt_resln_workspace(M, n))
            bufs += [dg, dbt, drs, dso, dws]
            L.check(c.lib.grl_gemm_nt_resln(c.ctx, B, M, n, K, dx.ptr, dw.ptr, db.ptr, dr.ptr, drs.ptr, dg.ptr, dbt.ptr, dy.ptr, eps, dso.ptr, dws.ptr), "gemm_nt_resln")
            ref = pre + (res[r] * rst[r, :1].astype(np.float64) - rst[r, 1:]) * (1 + b / 10) + sums / 10
            y, got_stats = c.download(dy, (M * n + 64,), B)[:M * n].reshape(M, n)[r].astype(np.float64), c.download(dso, (M, 2))[r]
            sd = np.sqrt(y.var(1) + eps)
            # single-pass moments in fp32 of n = 2040 values and eight partials: n / 8 * 2^-24 * (1 + (mean/sd)^2), doubled; the mean in units of sd
            assert np.abs(got_stats[:, 0] * sd - 1).max() < 1e-4 and np.abs(got_stats[:, 1] - y.mean(1) / sd).max() < 1e-4
        elif kind == "gated":
            L.check(c.lib.grl_swiglu_nt(c.ctx, B, B, M, n, K, dx.ptr, dw.ptr, dw.ptr, db.ptr, ds.ptr, dy.ptr, None, None), "swiglu_nt")
            up = O.truth_linear(x[r], w, sums)          # (any second bias)
            ref = pre * (up / (1 + np.exp(-up)))
        else:
            L.check(c.lib.grl_gemm_nt(c.ctx, B, out, M, n, K, dx.ptr, dw.ptr, db.ptr, dy.ptr, L.EPI_NONE), "gemm_nt")
            ref = pre
        got = c.download(dy, (M * n + 64,), out)
        assert (got[M * n:] == 7.0).all()
        assert O.max_rel(got[:M * n].reshape(M, n)[r], ref) < TOL_BF16
    finally:
        for t in bufs:
            t.free()


def poisoned(backend, kind, x, w, b, res, hit):
    """One product on 256 x 256 tiles; hit(x, w, res) plants its values first."""
    c, B, K, n = backend.core, L.GRL_BF16, x.shape[1], w.shape[0]
    m = x.shape[0]
    x, w, res = x.copy(), w.copy(), res.copy()
    hit(x, w, res)
    one = np.tile(np.array([0.9, 0.2], np.float32), (m, 1))
    cols = np.linspace(0.5, 1.5, n).astype(np.float32)
    dx, dw, db, dr, ds, dst, dy, dso, dws = bufs = [c.upload(x, B), c.upload(w, B), c.upload(b), c.upload(res, B), c.upload(cols), c.upload(one), c.alloc(m * n * 2),
                                                    c.alloc(m * 8), c.alloc(c.lib.grl_gemm_nt_resln_workspace(m, n))]
    try:
        if kind == "plain":
            L.check(c.lib.grl_gemm_nt(c.ctx, B, B, m, n, K, dx.ptr, dw.ptr, db.ptr, dy.ptr, L.EPI_NONE), "gemm_nt")
        elif kind == "folded":
            L.check(c.lib.grl_ln_gemm_nt_stats(c.ctx, B, B, m, n, K, dx.ptr, dw.ptr, ds.ptr, db.ptr, dst.ptr, dy.ptr, L.EPI_NONE), "ln_gemm_nt_stats")
        else:
            L.check(c.lib.grl_gemm_nt_resln(c.ctx, B, m, n, K, dx.ptr, dw.ptr, db.ptr, dr.ptr, dst.ptr, ds.ptr, db.ptr, dy.ptr, 1e-5, dso.ptr, dws.ptr), "gemm_nt_resln")
        return c.download(dy, (m, n), B), c.download(dso, (m, 2)) if kind == "normed_residual" else None
    finally:
        for t in bufs:
            t.free()


@pytest.mark.parametrize("kind", ["plain", "folded", "normed_residual"])
def test_infinities_and_nan_stay_in_their_rows_and_columns(backend, kind):
    """Rows, columns and residual elements that are not finite: those outputs are what IEEE makes of them, every other one keeps its bits."""
    rng = np.random.default_rng(3)
    K = 192
    x, w = O.bf16_round(rng.standard_normal((M, K), dtype=np.float32)), O.bf16_round((rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32))
    b, res = rng.standard_normal(N).astype(np.float32), O.bf16_round(rng.standard_normal((M, N), dtype=np.float32))
    x[x == 0] = 1.0
    w[w == 0] = 1.0
    nan_row, inf_row, col, at = 300, M - 1, 261, (7000, 1999)
    x[:, 5] = np.abs(x[:, 5])

    def hit(x, w, res):
        x[nan_row, 70], x[inf_row, 191] = np.nan, -np.inf
        w[col, 5] = np.inf
        res[at] = -np.inf
    clean, clean_stats = poisoned(backend, kind, x, w, b, res, lambda *a: None)
    got, stats = poisoned(backend, kind, x, w, b, res, hit)
    assert np.isfinite(clean).all()
    assert np.isnan(got[nan_row]).all()
    others = np.arange(N) != col
    np.testing.assert_array_equal(got[inf_row, others], (-np.inf * np.sign(w[others, 191])).astype(np.float32))
    rows = np.ones(M, bool)
    rows[[nan_row, inf_row]] = False
    assert (got[rows, col] == np.inf).all()
    keep = rows[:, None] & others[None, :]
    if kind == "normed_residual":
        assert got[at] == -np.inf
        keep[at] = False
    np.testing.assert_array_equal(got[keep], clean[keep])


def test_folded_rows_far_from_zero(backend):
    """Row means eight spreads from zero: the epilogue takes mean * column sum off the raw product."""
    rng = np.random.default_rng(8)
    K = 768
    x, W, b, g, bt = lnl.make(rng, M, K, N, mean=8.0)
    x, W, r = O.bf16_round(x), O.bf16_round(W), rows_of(rng)
    y = lnl.ln_linear(backend, "bf16", x, g, bt, W, b, 1e-5)[0]
    assert np.isfinite(y).all()
    assert O.max_rel(y[r], O.truth_linear(O.truth_layernorm(x[r], g, bt, 1e-5), W, b)) < TOL_BF16


@pytest.mark.parametrize("slabs", [2, 5])
def test_residual_of_fp32_results(backend, slabs):
    """bf16 operands, an fp32 residual and fp32 results (in place): every unit of a tile's output gets its own residual.  Tolerance: fp32 sums
    of K products, 2^-23 * K of the largest."""
    c, B, K = backend.core, L.GRL_BF16, 64 * slabs
    rng = np.random.default_rng(slabs)
    x, w = O.bf16_round(rng.standard_normal((M, K), dtype=np.float32)), O.bf16_round((rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32))
    b, res, r = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N), dtype=np.float32), rows_of(rng)
    bufs = [c.upload(x, B), c.upload(w, B), c.upload(b), c.upload(res)]
    try:
        dx, dw, db, dy = bufs
        L.check(c.lib.grl_gemm_nt_res(c.ctx, B, L.GRL_F32, M, N, K, dx.ptr, dw.ptr, db.ptr, dy.ptr, dy.ptr), "gemm_nt_res")
        ref = O.truth_linear(x[r], w, b) + res[r].astype(np.float64)
        assert O.max_rel(c.download(dy, (M, N))[r], ref) < K * 2.0 ** -23
    finally:
        for t in bufs:
            t.free()


@pytest.mark.parametrize("slabs", [2, 3, 7])
@pytest.mark.parametrize("kind", ["residual", "normed_residual"])
def test_one_tile_for_each_unit(backend, monkeypatch, kind, slabs):
    """213 tiles: the residual's lines are asked for under the last steps, also where those are the first"""
    monkeypatch.setitem(globals(), "M", 71 * 256 - 37)
    monkeypatch.setitem(globals(), "N", 3 * 256 - 8)
    test_phased_tiles(backend, kind, slabs)
