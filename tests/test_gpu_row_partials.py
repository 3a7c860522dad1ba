"""GPU parity of row statistics that stay partial sums between products: several folded layers in one call against the same layers one
call each (which merge them in a launch of their own), and the gated MLP block against its two products.  Widths give 1 to 6 partials, and
7 and more, which are merged in any case; row counts, odd ones among them, reach every kernel that writes or reads them in bf16 (64 x 64 and
64 x 128 tiles, 128 x 128 on four and eight waves, 256 x 256 with more than one tile per workgroup, and the small ones that take none) with
ragged last tiles.  The kernels' numbers stand beside the sizes; test_dispatch_host.py holds them against the launchers' rules.
The sums are the same in the same order, so what differs is at most the rounding of a quotient: 2^-23 of a statistic, which can move a
stored value by one unit of its type (bf16 2^-8, fp32 2^-23) and that unit through the rest: 2-norms agree to 4e-3 and 4e-6."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT
from grilly_amd import _lib as L

pytestmark = pytest.mark.gpu

NEAR = {"bf16": 4e-3, "fp32": 4e-6}


def near(a, b, dtype):
    a, b = a.astype(np.float64), b.astype(np.float64)
    assert np.isfinite(a).all()
    assert np.linalg.norm(a - b) <= NEAR[dtype] * np.linalg.norm(b)


# (sequences, length, heads of 64, d_ff, bf16 kernels of out-proj, FFN2 (these write partials), QKV, FFN1 (these read them))
LAYERS = [(1, 1, 2, 64, (7, 7, 9, 9)), (3, 43, 2, 192, (7, 7, 9, 9)), (5, 60, 6, 256, (7, 7, 9, 9)), (20, 65, 12, 192, (7, 7, 6, 9)), (21, 120, 12, 448, (7, 7, 4, 8)),
          (70, 128, 6, 1536, (6, 6, 4, 3)), (90, 160, 12, 256, (4, 4, 4, 6)), (9, 100, 14, 128, (7, 7, 6, 9)), (13, 100, 16, 128, (7, 7, 4, 9)),
          (19, 67, 12, 192, (7, 7, 6, 9)), (73, 73, 12, 256, (6, 6, 4, 8)), (85, 511, 12, 768, (3, 3, 3, 3))]


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("B,S,heads,ff", [l[:4] for l in LAYERS])
def test_layers_in_one_call(backend, dtype, B, S, heads, ff):
    import grilly_amd
    c, d = backend.core, 64 * heads
    cfg = grilly_amd.EncoderConfig(layers=3, d_model=d, heads=heads, d_ff=ff, vocab=200, max_pos=512)
    w = grilly_amd.random_bert_weights(cfg, seed=B + S)
    rng = np.random.default_rng(B * S)
    for lw in w["layers"]:
        for k in lw:
            if not k.startswith("w_"):
                lw[k] = (lw[k] + 0.1 * rng.standard_normal(lw[k].shape)).astype(np.float32)
    enc = grilly_amd.BertEncoder(backend, cfg, w, dtype=dtype, fused=True)
    ids = rng.integers(0, 200, (B, S))
    mask = (np.arange(S) < rng.integers(1, S + 1, B)[:, None]).astype(np.int64)
    got = enc.forward(ids, mask, pool=False)
    lib = c.lib
    enc.set_inputs(ids, mask)
    L.check(lib.grl_embed(c.ctx, enc.code, B, S, d, cfg.vocab, enc.ids.ptr, enc.tok.ptr, enc.pos.ptr, enc.typ.ptr, enc.x.ptr), "embed")
    L.check(lib.grl_ln_stats(c.ctx, enc.code, B * S, d, enc.x.ptr, cfg.embedding_eps, enc.stats.ptr), "stats")
    for f in enc.fused_structs:
        L.check(lib.grl_bert_layer_fwd_fused(c.ctx, enc.code, B, S, heads, cfg.head_dim, ff, ctypes.byref(f), enc.mask.ptr, cfg.eps, enc.x.ptr,
                                             enc.stats.ptr, enc.ws.ptr), "layer")
    enc._last_layernorm(B * S)
    near(got, c.download(enc.x, (B, S, d), enc.code), dtype)
    enc.release_activations()


# (rows, d_model, d_ff, bf16 kernels of the product that writes partials and of the gated one)
GATED = [(1, 64, 64, 7, 9), (130, 384, 96, 7, 9), (1400, 768, 200, 7, 10), (3100, 768, 1152, 6, 4), (7300, 640, 1152, 4, 4), (26000, 768, 1152, 4, 3), (900, 960, 128, 7, 9),
         (2501, 384, 384, 7, 10), (2501, 768, 384, 7, 10), (9001, 384, 384, 6, 4), (5001, 768, 384, 6, 4), (11001, 384, 384, 4, 4), (7301, 768, 384, 4, 4),
         (43435, 768, 384, 3, 3), (32695, 1024, 512, 3, 3)]


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("M,d,ff", [g[:3] for g in GATED])
def test_gated_block(backend, dtype, M, d, ff):
    c, code, lib = backend.core, (L.GRL_BF16 if dtype == "bf16" else L.GRL_F32), backend.core.lib
    rng = np.random.default_rng(M + d)
    f = lambda *s: rng.standard_normal(s, dtype=np.float32)
    up, upw = (lambda a: c.upload(a)), (lambda a: c.upload(a, code))
    A, W, R, Wg, Wu = upw(f(M, d)), upw(f(d, d) * 0.05), upw(f(M, d) + 0.5), upw(f(ff, d) * 0.05), upw(f(ff, d) * 0.05)
    b, g, bt, cg, cu, bg, bu = up(f(d)), up(1 + 0.1 * f(d)), up(f(d)), up(f(ff)), up(f(ff)), up(f(ff)), up(f(ff))
    st = c.upload_raw(np.stack([np.full(M, 0.9, np.float32), np.full(M, 0.3, np.float32)], 1).copy())
    es = 2 if dtype == "bf16" else 4
    C1, C2, o1, o2, stats = c.alloc(M * d * es), c.alloc(M * d * es), c.alloc(M * ff * es), c.alloc(M * ff * es), c.alloc(M * 8 + 16)
    ws = c.alloc(int(lib.grl_gemm_nt_resln_workspace(M, d)))
    L.check(lib.grl_resln_ln_glu(c.ctx, code, M, d, d, ff, A.ptr, W.ptr, b.ptr, R.ptr, st.ptr, g.ptr, bt.ptr, C1.ptr, Wg.ptr, Wu.ptr, cg.ptr, cu.ptr, bg.ptr, bu.ptr,
                                 1e-5, stats.ptr, ws.ptr, o1.ptr, L.EPI_GELU), "resln_ln_glu")
    L.check(lib.grl_gemm_nt_resln(c.ctx, code, M, d, d, A.ptr, W.ptr, b.ptr, R.ptr, st.ptr, g.ptr, bt.ptr, C2.ptr, 1e-5, stats.ptr, ws.ptr), "resln")
    L.check(lib.grl_ln_glu_nt_stats(c.ctx, code, code, M, ff, d, C2.ptr, Wg.ptr, Wu.ptr, cg.ptr, cu.ptr, bg.ptr, bu.ptr, stats.ptr, o2.ptr, L.EPI_GELU), "glu")
    np.testing.assert_array_equal(c.download(C1, (M, d), code), c.download(C2, (M, d), code))
    near(c.download(o1, (M, ff), code), c.download(o2, (M, ff), code), dtype)
    for t in (A, W, R, Wg, Wu, b, g, bt, cg, cu, bg, bu, st, C1, C2, o1, o2, stats, ws):
        t.free()


FORCED = """
import sys
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
import grilly_amd, test_gpu_row_partials as t
backend = grilly_amd.Compute()
for dtype in ("fp32", "bf16"):
    for shape in ((130, 384, 96), (1401, 768, 200)):
        print(dtype, shape, flush=True)
        t.test_gated_block(backend, dtype, *shape)
print("passed")
"""


@pytest.mark.parametrize("variant", [6, 7, 8])
def test_gated_block_with_a_forced_kernel(variant):
    """GRL_GEMM_VARIANT may name a kernel that a two-weight product does not have: the one that runs in its place takes no partials."""
    child = subprocess.run([sys.executable, "-c", FORCED, ROOT], capture_output=True, text=True, timeout=100, env=dict(os.environ, GRL_GEMM_VARIANT=str(variant)))
    assert child.returncode == 0 and "passed" in child.stdout, child.stdout + child.stderr
