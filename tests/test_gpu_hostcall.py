"""Operators on host arrays: the sizes where the path changes (one pinned slab / rings and blocks, results written in place /
copied back in one piece or in chunks), transfers of odd byte counts, results that are kept, and calls from several threads."""
import os
import threading

import numpy as np
import pytest

from conftest import TOL_F32, TOL_BF16
from oracle import oracle_np as O
from grilly_amd import _lib as L

pytestmark = pytest.mark.gpu


# (M, K, N): 64 KiB of results in place and just above; 2 MiB and just above; several blocks of rows with a ragged last
# one; rows that are no multiple of 16 bytes; one row of a wide product; more blocks than there are rows for
# and, around the 5 MiB up to which a call is one slab: inputs of several parts with a ragged last one, odd widths, one row more
SLAB_SHAPES = [(900, 384, 517), (3, 1100, 1101), (520, 1025, 300), (2431, 256, 256), (2432, 256, 256), (1250, 384, 700)]
SHAPES = [(128, 64, 128), (130, 64, 128), (700, 384, 128), (710, 384, 128), (9001, 256, 640), (4099, 40, 1030), (1, 2048, 4096), (17, 4096, 24000)]


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("M,K,N", SHAPES + SLAB_SHAPES)
def test_linear_on_host_arrays(backend, dtype, M, K, N):
    rng = np.random.default_rng(M + N)
    x = rng.standard_normal((M, K), dtype=np.float32)
    w = rng.standard_normal((N, K), dtype=np.float32) * np.float32(1 / np.sqrt(K))
    b = rng.standard_normal(N, dtype=np.float32)
    xs, keep = (O.bf16_round(x), O.bf16_round(w)) if dtype == "bf16" else (x, w), (x.copy(), w.copy())
    y = backend.fnn.linear(x, w, b, dtype=dtype)
    assert y.shape == (M, N) and y.dtype == np.float32 and y.flags.c_contiguous and y.flags.writeable
    rows = np.unique(np.concatenate([np.arange(min(M, 3)), np.arange(max(M - 3, 0), M), rng.integers(0, M, 40)]))
    ref = O.truth_linear(xs[0][rows], xs[1], b)
    assert O.max_rel(y[rows], ref) < (TOL_F32 if dtype == "fp32" else TOL_BF16)
    assert np.isfinite(y).all()
    np.testing.assert_array_equal(x, keep[0])
    np.testing.assert_array_equal(w, keep[1])


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("B,S,masked", [(3, 40, True), (12, 100, True), (40, 128, True), (37, 200, False), (1, 2100, False)])
def test_attention_on_host_arrays(backend, dtype, B, S, masked):
    H, D = 4, 64
    rng = np.random.default_rng(B + S)
    q, k, v = (O.bf16_round(rng.standard_normal((B, S, H, D)).astype(np.float32)) for _ in range(3))
    mask = (np.arange(S) < rng.integers(1, S + 1, B)[:, None]).astype(np.float32) if masked else None
    o = backend.attention.flash_attention2(q, k, v, H, D, mask=mask, dtype=dtype)
    for b in {0, B // 2, B - 1}:
        ref = O.truth_attention(q[b:b + 1], k[b:b + 1], v[b:b + 1], mask=None if mask is None else mask[b:b + 1])
        assert O.max_rel(o[b:b + 1], ref) < (TOL_F32 if dtype == "fp32" else TOL_BF16)


@pytest.mark.parametrize("nbytes", [1, 7, 4096, (256 << 10) - 1, (256 << 10) + 4, (3 << 20) + 5, 33 << 20])
def test_transfers_are_exact(backend, nbytes):
    c = backend.core
    src = np.random.default_rng(nbytes).integers(0, 256, nbytes, dtype=np.uint8)
    dst = np.zeros(nbytes + 8, np.uint8)
    with c.alloc(nbytes + 16) as d:
        for off in (0, 3):
            L.check(c.lib.grl_h2d(c.ctx, d.ptr + off, src.ctypes.data, nbytes))
            L.check(c.lib.grl_d2h(c.ctx, dst.ctypes.data, d.ptr + off, nbytes))
            np.testing.assert_array_equal(dst[:nbytes], src)
            assert not dst[nbytes:].any()
            dst[:] = 0


@pytest.mark.parametrize("n", [5, 131072, 131073, 3000001])
def test_bf16_transfers_round_to_nearest_even(backend, n):
    x = np.random.default_rng(n).integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32).view(np.float32)
    x[:4] = [np.nan, np.inf, -np.inf, -0.0]
    c = backend.core
    buf = c.upload(x, L.GRL_BF16)
    got = c.download(buf, (n,), L.GRL_BF16)
    buf.free()
    u = x.view(np.uint32)
    want = np.where((u & 0x7fffffff) > 0x7f800000, (u >> 16) | 0x40, (u + 0x7fff + ((u >> 16) & 1)) >> 16).astype(np.uint32) << 16
    np.testing.assert_array_equal(got.view(np.uint32), want)


def test_kept_results_stay_what_they_were(backend):
    """Results of a program that keeps them are its own: more of them than wait for reuse (512 MiB), views that outlive their
    array, and none changed by later calls."""
    n = 1 << 24                                      # 64 MiB each
    kept = []
    for i in range(10):
        y = backend.fnn.residual(np.full(n, i, np.float32), np.full(n, 0.5, np.float32))
        kept.append(y[n // 2:n // 2 + 4] if i % 2 else y)
        del y
    for i, y in enumerate(kept):
        assert (y == i + 0.5).all()


def test_large_calls_from_several_threads(backend):
    errors = []

    def worker(t):
        try:
            rng = np.random.default_rng(t)
            x = rng.standard_normal((3000 + 100 * t, 256), dtype=np.float32)
            w = rng.standard_normal((512, 256), dtype=np.float32)
            small = rng.standard_normal((8, 256), dtype=np.float32)
            want, want_small = x @ w.T, small @ w.T
            for _ in range(6):
                assert O.max_rel(backend.fnn.linear(x, w), want) < TOL_F32
                assert O.max_rel(backend.fnn.linear(small, w), want_small) < TOL_F32
        except Exception as e:
            errors.append((t, repr(e)))

    threads = [threading.Thread(target=worker, args=(t,)) for t in range(5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not errors and not any(t.is_alive() for t in threads)


def test_results_are_the_callers_own(backend):
    """A large result is an array like any other: numpy owns and resizes it, a forked child reads it and has its own copy of
    it, and a program that trims gets the memory of collected results back."""
    n = 3 << 22                                      # 48 MiB
    def result(v):
        return backend.fnn.residual(np.full(n, v, np.float32), np.full(n, 0.5, np.float32))

    y = result(3)
    assert y.flags.owndata and y.base is None
    for size in (n // 3, n):
        y.resize(size, refcheck=False)
        assert y.shape == (size,) and (y[:n // 3] == 3.5).all()
    y = result(4)
    child = os.fork()
    if child == 0:
        good = bool((y == 4.5).all())
        y[:] = 7.0
        z = np.empty(n, np.float32)
        z[:] = y
        os._exit(0 if good and (z == 7.0).all() else 1)
    assert os.waitpid(child, 0)[1] == 0
    assert (y == 4.5).all()

    def resident():
        return int(open("/proc/self/statm").read().split()[1]) * 4096

    del y
    before = resident()
    L.check(backend.core.lib.grl_pool_trim(backend.core.ctx))
    assert resident() <= before - n * 4
