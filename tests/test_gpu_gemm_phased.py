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
@pytest.mark.parametrize("kind", ["gelu", "residual", "folded", "gated", "f32_out", "odd_columns"])
def test_phased_tiles(backend, kind, slabs):
    c, B, K = backend.core, L.GRL_BF16, 64 * slabs
    rng = np.random.default_rng(slabs)
    q = lambda a: O.bf16_round(a.astype(np.float32))
    n = N - 3 if kind == "odd_columns" else N // 2 if kind == "gated" else N
    x, w, b, r = q(rng.standard_normal((M, K), dtype=np.float32) + 0.5), q(rng.standard_normal((n, K)) / np.sqrt(K)), rng.standard_normal(n).astype(np.float32), rows_of(rng)
    res = q(rng.standard_normal((M, n), dtype=np.float32)) if kind == "residual" else np.zeros((1, n), np.float32)
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
