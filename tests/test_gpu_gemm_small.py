"""GPU parity of the GEMM kernels for products that 128 x 128 tiles leave short of work, against the float64 oracle: tiles whose K
slabs the four waves share out (32 x 32 and 64 x 64), and the rings of three and four LDS stages (64 x 64, 64 x 128, 128 x 128).
Sizes sit where these can go wrong: fewer K slabs than waves or stages, slab counts that do not divide by either, one row,
one column group, ragged last tiles, and the sizes on either side of a dispatch line.
Tolerances: max|y-ref|/max|ref| <= 1e-4 (fp32), <= 2e-2 (bf16), as in the other GEMM tests."""
import numpy as np
import pytest

import test_gpu_fused_layer as fused_layer
import test_gpu_ln_linear as lnl
from conftest import TOL_F32, TOL_BF16
from oracle import oracle_np as O
from grilly_amd import _lib as L

pytestmark = pytest.mark.gpu

TOL = {"fp32": TOL_F32, "bf16": TOL_BF16}
CODE = {"fp32": L.GRL_F32, "bf16": L.GRL_BF16}

# (M, slabs of 128 bytes, N)
PLAIN = [(1, 1, 4), (33, 5, 36), (128, 12, 2304), (250, 48, 768), (30, 70, 100),          # 32 x 32 tiles (the last: split K in fp32)
         (800, 12, 768), (777, 13, 780), (1990, 97, 764),                                 # bf16: 64 x 64 shared K, one and two per compute unit
         (450, 1, 3072), (449, 2, 3004), (449, 3, 3072), (450, 13, 3072),                 # 64 x 64 ring around its four stages
         (1500, 1, 2304), (1499, 2, 2300), (1500, 3, 2304), (1500, 4, 2304), (1500, 5, 2304),   # bf16: 128 x 128 ring
         (3000, 1, 1152), (2999, 2, 1148), (3000, 3, 1152), (3000, 12, 1152)]             # fp32: 64 x 128 ring


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("M,slabs,N", PLAIN)
def test_plain_gelu_residual(backend, dtype, M, slabs, N):
    c, code = backend.core, CODE[dtype]
    K = slabs * (64 if dtype == "bf16" else 32)
    rng = np.random.default_rng(M + 3 * K + 7 * N)
    q = lambda a: lnl.q(dtype, a.astype(np.float32))
    x, W, r = q(rng.standard_normal((M, K))), q(rng.standard_normal((N, K)) / np.sqrt(K)), q(2 * rng.standard_normal((M, N)))
    b = rng.standard_normal(N).astype(np.float32)
    es, pad = (2 if dtype == "bf16" else 4), 64
    guard = np.full(M * N + pad, 7.0, np.float32)              # stores past the matrix show up behind it
    bufs = [c.upload(x, code), c.upload(W, code), c.upload(b), c.upload(r, code), c.upload(guard, code)]
    dx, dw, db, dr, dy = bufs
    try:
        for bias, pb in ((b, db.ptr), (None, None)):
            pre = O.truth_linear(x, W, bias)
            L.check(c.lib.grl_gemm_nt(c.ctx, code, code, M, N, K, dx.ptr, dw.ptr, pb, dy.ptr, L.EPI_NONE), "gemm_nt")
            got = c.download(dy, (M * N + pad,), code)
            assert O.max_rel(got[:M * N].reshape(M, N), pre) < TOL[dtype] and (got[M * N:] == 7.0).all()
            L.check(c.lib.grl_gemm_nt(c.ctx, code, code, M, N, K, dx.ptr, dw.ptr, pb, dy.ptr, L.EPI_GELU), "gemm_nt gelu")
            got = c.download(dy, (M, N), code)
            assert O.max_rel(got, O.truth_gelu(pre)) < TOL[dtype]
        L.check(c.lib.grl_gemm_nt_res(c.ctx, code, code, M, N, K, dx.ptr, dw.ptr, db.ptr, dr.ptr, dr.ptr), "gemm_nt_res")      # in place
        assert O.max_rel(c.download(dr, (M, N), code), O.truth_linear(x, W, b) + r.astype(np.float64)) < TOL[dtype]
    finally:
        for t in bufs:
            t.free()


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("M,K,N", [(1, 64, 4), (130, 320, 1152), (450, 768, 1148), (800, 768, 768), (1500, 192, 2304), (3000, 384, 1152)])
def test_folded_layernorm(backend, dtype, M, K, N):
    rng = np.random.default_rng(M + K + N)
    x, W, b, g, bt = lnl.make(rng, M, K, N)
    x, W = lnl.q(dtype, x), lnl.q(dtype, W)
    ref = O.truth_layernorm(x, g, bt, 1e-5)
    assert O.max_rel(lnl.ln_linear(backend, dtype, x, g, bt, W, b, 1e-5)[0], O.truth_linear(ref, W, b)) < TOL[dtype]
    if N <= 1152:
        Wu, bu = lnl.q(dtype, W[::-1].copy()), b[::-1].copy()
        y = lnl.ln_glu(backend, dtype, x, g, bt, W, Wu, b, bu, 1e-5, "gelu")
        assert O.max_rel(y, O.truth_linear(ref, W, b) * O.truth_gelu(O.truth_linear(ref, Wu, bu))) < TOL[dtype]


# tiles of 64 and of 128 rows; fewer slabs than stages; ragged rows and columns
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("M,K,N", [(1, 64, 768), (2499, 64, 768), (2500, 192, 760), (2900, 128, 768), (2899, 256, 768), (3000, 448, 384)])
def test_layernormed_residual(backend, dtype, M, K, N):
    fused_layer.test_gemm_with_layernormed_residual_and_row_statistics(backend, dtype, False, M, K, N)


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("M,K,N", [(3000, 768, 768), (700, 768, 768), (4000, 256, 1024), (16384, 128, 2048)])
def test_blocks_of_a_host_call_add_in_the_order_of_the_whole_product(backend, dtype, M, K, N):
    c, code = backend.core, CODE[dtype]
    rng = np.random.default_rng(M + N)
    x, W = lnl.q(dtype, rng.standard_normal((M, K)).astype(np.float32)), lnl.q(dtype, rng.standard_normal((N, K)).astype(np.float32))
    b = rng.standard_normal(N).astype(np.float32)
    dx, dw, db, dy = bufs = [c.upload(x, code), c.upload(W, code), c.upload(b), c.alloc(M * N * 4)]
    try:
        L.check(c.lib.grl_gemm_nt(c.ctx, code, code, M, N, K, dx.ptr, dw.ptr, db.ptr, dy.ptr, L.EPI_NONE), "gemm_nt")
        np.testing.assert_array_equal(backend.fnn.linear(x, W, b, dtype=dtype), c.download(dy, (M, N), code))
    finally:
        for t in bufs:
            t.free()
