"""Batches without their padding (grl_ragged): the native packing pass, attention over sequences stored back to back
against the float64 oracle sequence by sequence, and the encoders' pooled forward against their own rectangular form."""
import ctypes

import numpy as np
import pytest

from conftest import TOL_F32, TOL_BF16
from oracle import oracle_np as O
from grilly_amd import (BertEncoder, EncoderConfig, PreNormEncoder, PreNormEncoderConfig, random_bert_weights, random_prenorm_weights)
from grilly_amd import _lib as L


def pack(ids, mask, vocab=100):
    B, S = ids.shape
    out = np.full(B + 1 + 2 * B * S, -7, np.int32)
    rows, longest = ctypes.c_int64(), ctypes.c_int64()
    kind = 0 if mask is None else 1 if mask.dtype == np.int64 else 2
    rc = L.load().grl_pack_batch(B, S, vocab, ids.ctypes.data, None if mask is None else mask.ctypes.data, kind, out.ctypes.data,
                                 ctypes.byref(rows), ctypes.byref(longest))
    n = rows.value
    return rc, out[:B + 1], out[B + 1:B + 1 + n], out[B + 1 + n:B + 1 + 2 * n], longest.value


@pytest.mark.parametrize("form", ["none", "right", "left", "holes", "empty", "int64"])
def test_pack_batch(form):
    rng = np.random.default_rng(5)
    B, S = 5, 13
    ids = rng.integers(0, 100, (B, S))
    n = np.array([13, 1, 7, 12, 4])
    keep = {"none": np.ones((B, S), bool), "right": np.arange(S) < n[:, None], "left": np.arange(S) >= S - n[:, None],
            "holes": rng.random((B, S)) < 0.5, "empty": np.arange(S) < np.array([0, 3, 0, 13, 0])[:, None],
            "int64": np.arange(S) < n[:, None]}[form]
    mask = None if form == "none" else keep.astype(np.int64 if form == "int64" else np.float32)
    rc, off, pos, kept, longest = pack(ids, mask)
    assert rc == (L.PACK_SCATTERED if form in ("left", "holes") else L.PACK_PREFIX)
    np.testing.assert_array_equal(off, np.concatenate([[0], np.cumsum(keep.sum(1))]))
    np.testing.assert_array_equal(pos, np.nonzero(keep)[1])
    np.testing.assert_array_equal(kept, ids[keep])
    assert longest == keep.sum(1).max()


def test_pack_batch_refusals():
    ids = np.zeros((2, 3), np.int64)
    assert pack(ids, np.array([[1, 1, 0.5], [1, 0, 0]], np.float32))[0] == L.PACK_OTHER_MASK
    assert pack(ids, np.array([[1, np.nan, 0], [1, 0, 0]], np.float32))[0] == L.PACK_OTHER_MASK
    bad = ids.copy()
    bad[1, 2] = 100                                    # a padded position counts too
    assert pack(bad, np.array([[1, 1, 0], [1, 0, 0]], np.float32))[0] == L.PACK_BAD_ID
    bad[1, 2] = -1
    assert pack(bad, None)[0] == L.PACK_BAD_ID
    assert L.load().grl_pack_batch(2, 3, 0, None, None, 0, None, None, None) == L.ERR_SHAPE
    assert L.load().grl_fa2_fwd_ragged(None, 0, None, 1, 32, None, None, None, None, 32, 32, 32, 32, 1.0, 0, 0, 1.0, 1.0) == L.ERR_ARG


# edges of the 32-query waves, 64- and 128-key tiles and 128- / 256-query workgroups, an empty and a one-token sequence
# and enough sequences (of two heads each, no whole turn of eight) that their heads are dealt out
LENGTHS = {"short": [1, 32, 0, 33, 64, 65, 127, 129], "long": [1025, 3, 256, 1200], "many": [(37 * i * i + 11 * i) % 290 for i in range(35)]}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("lengths", sorted(LENGTHS))
@pytest.mark.parametrize("D,causal,rope", [(32, False, None), (64, False, "half"), (64, True, "interleaved"), (128, True, "half"), (48, False, "half")])
def test_fa2_ragged(backend, dtype, lengths, D, causal, rope):
    c, H, lens = backend.core, 2, LENGTHS[lengths]
    code = L.GRL_BF16 if dtype == "bf16" else L.GRL_F32
    rng = np.random.default_rng(D + len(lens))
    rows = sum(lens)
    q, k, v = (rng.standard_normal((rows, H, D)).astype(np.float32) for _ in range(3))
    if dtype == "bf16":
        q, k, v = (O.bf16_round(t) for t in (q, k, v))
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    pos = np.concatenate([np.arange(n) for n in lens]).astype(np.int32)
    dq, dk, dv, do, dp = c.upload(q, code), c.upload(k, code), c.upload(v, code), c.upload_raw(off), c.upload_raw(pos)
    out = c.alloc(rows * H * D * 4)
    style = {None: L.ROPE_NONE, "half": L.ROPE_HALF, "interleaved": L.ROPE_INTERLEAVED}[rope]
    try:
        rg = L.Ragged(do.ptr, dp.ptr, len(lens), rows, max(lens))
        L.check(c.lib.grl_fa2_fwd_ragged(c.ctx, code, ctypes.byref(rg), H, D, dq.ptr, dk.ptr, dv.ptr, out.ptr, H * D, H * D, H * D, H * D,
                                         1.0 / float(np.sqrt(D)), int(causal), style, 10000.0, 1.0), "fa2_ragged")
        o = c.download(out, (rows, H, D), code)
    finally:
        for t in (dq, dk, dv, do, dp, out):
            t.free()
    for b, n in enumerate(lens):
        if n:
            s = slice(off[b], off[b + 1])
            ref = O.truth_attention(q[None, s], k[None, s], v[None, s], causal=causal, rope=rope)
            assert O.max_rel(o[None, s], ref) < (TOL_F32 if dtype == "fp32" else TOL_BF16), (b, n)


# just inside and just outside the rule that ranks the sequences by length: 640 blocks of 128 queries at least, 32 sequences at most, longer than 256
@pytest.mark.gpu
@pytest.mark.parametrize("D,H,causal,lens", [
    (64, 8, False, [257] + [1] * 30 + [256]), (64, 9, False, [0, 300, 300, 17, 0] + [300] * 20), (64, 12, True, [500] + list(range(3, 500, 29))),
    (128, 8, False, [400 - 9 * i for i in range(32)]), (64, 8, False, [300 - 9 * i for i in range(33)]), (64, 40, False, [900, 1, 899])])
def test_order_of_sequences(backend, D, H, causal, lens):
    """Where a sequence stands in the batch changes nothing but where its result stands: bit for bit, and against the oracle."""
    c, rng, scale = backend.core, np.random.default_rng(D + len(lens)), 1.0 / float(np.sqrt(D))
    parts = [[O.bf16_round(rng.standard_normal((n, H, D)).astype(np.float32)) for _ in range(3)] for n in lens]

    def run(order):
        off = np.concatenate([[0], np.cumsum([lens[i] for i in order])]).astype(np.int32)
        pos = np.concatenate([np.arange(lens[i]) for i in order]).astype(np.int32)
        bufs = [c.upload(np.concatenate([parts[i][j] for i in order]), L.GRL_BF16) for j in range(3)] + [c.upload_raw(off), c.upload_raw(pos), c.alloc(int(off[-1]) * H * D * 2)]
        try:
            rg = L.Ragged(bufs[3].ptr, bufs[4].ptr, len(lens), int(off[-1]), max(lens))
            L.check(c.lib.grl_fa2_fwd_ragged(c.ctx, L.GRL_BF16, ctypes.byref(rg), H, D, bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, bufs[5].ptr, H * D, H * D, H * D, H * D,
                                             scale, int(causal), L.ROPE_NONE, 10000.0, 1.0), "fa2_ragged")
            o = c.download(bufs[5], (int(off[-1]), H, D), L.GRL_BF16)
        finally:
            for t in bufs:
                t.free()
        return {i: o[off[k]:off[k + 1]] for k, i in enumerate(order)}

    one, other = run(list(range(len(lens)))), run([int(i) for i in rng.permutation(len(lens))])
    for i, n in enumerate(lens):
        np.testing.assert_array_equal(one[i], other[i])
        if n:
            assert O.max_rel(one[i][None], O.truth_attention(*(t[None] for t in parts[i]), causal=causal)) < TOL_BF16, (i, n)


# batches that the rule ranks, with empty sequences, equal lengths and causal ones; the last just past its line for full rectangles
@pytest.mark.gpu
@pytest.mark.parametrize("D,H,causal,lens", [
    (64, 9, False, [0, 300, 300, 17, 0] + [300] * 10 + [100] * 12), (64, 12, True, [600] + list(range(3, 600, 35))), (128, 8, True, [0, 700, 699, 1] + [350] * 12),
    (64, 10, False, [400] * 17 + [0] * 6), (64, 10, False, [400] * 17 + [0] * 5)])
def test_order_of_unequal_sequences(backend, D, H, causal, lens):
    test_order_of_sequences(backend, D, H, causal, lens)


def _masks(rng, B, S):
    n = rng.integers(1, S + 1, B)
    n[0] = S
    right = (np.arange(S) < n[:, None]).astype(np.int64)
    gone = right.copy()
    gone[1] = 0
    return {"right": right, "left": right[:, ::-1].copy(), "holes": (rng.random((B, S)) < 0.6).astype(np.float32), "one_empty": gone,
            "soft": np.where(right > 0, 1.0, 0.25).astype(np.float32)}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("arch,fused", [("bert", False), ("bert", True), ("prenorm", None)])
@pytest.mark.parametrize("form", ["right", "left", "holes", "one_empty", "soft"])
def test_pooled_forward_without_padding(backend, dtype, arch, fused, form):
    """forward(pool=True) against launch() on the same ids and mask, which computes the padding as well.  The two run the
    same arithmetic on other row counts (other tiles, other groupings of partial sums): rounding only, 1e-5 in fp32; in bf16
    two layers round each state about a dozen times at 2^-9 each, 2^-9 * sqrt(12) = 7e-3 of its size."""
    B, S = 6, 75
    rng = np.random.default_rng(11)
    if arch == "bert":
        cfg = EncoderConfig(layers=2, d_model=128, heads=2, d_ff=256, vocab=300, max_pos=S)
        enc = BertEncoder(backend, cfg, random_bert_weights(cfg, seed=2, std=0.08), dtype=dtype, fused=fused)
    else:
        cfg = PreNormEncoderConfig(layers=2, d_model=128, heads=2, d_ff=192, vocab=300)
        enc = PreNormEncoder(backend, cfg, random_prenorm_weights(cfg, seed=2, std=0.08), dtype=dtype)
    ids = rng.integers(0, 300, (B, S))
    mask = _masks(rng, B, S)[form]
    got = enc.forward(ids, mask)
    enc.set_inputs(ids, mask)
    enc.launch(True)
    want = backend.core.download(enc.pooled, (B, cfg.d_model))
    assert O.max_rel(got, want) < (1e-5 if dtype == "fp32" else 7e-3)
    # a mask of ones is the same batch as no mask, bit for bit
    np.testing.assert_array_equal(enc.forward(ids, np.ones((B, S), np.int64)), enc.forward(ids, None))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("arch", ["bert", "prenorm"])
@pytest.mark.parametrize("form", ["right", "left", "holes", "soft", "none"])
def test_launch_after_a_pooled_forward(backend, dtype, arch, form):
    """launch() runs the batch that forward() had last, whatever form that forward took: the same kernels on the same inputs
    as after set_inputs(), so the same bits.  The batch before has the same shape and another mask, or none."""
    B, S = 6, 75
    rng = np.random.default_rng(12)
    if arch == "bert":
        cfg = EncoderConfig(layers=2, d_model=128, heads=2, d_ff=256, vocab=300, max_pos=S)
        enc = BertEncoder(backend, cfg, random_bert_weights(cfg, seed=3, std=0.08), dtype=dtype)
    else:
        cfg = PreNormEncoderConfig(layers=2, d_model=128, heads=2, d_ff=192, vocab=300)
        enc = PreNormEncoder(backend, cfg, random_prenorm_weights(cfg, seed=3, std=0.08), dtype=dtype)
    masks = _masks(rng, B, S)
    mask = masks.get(form)
    ids, before = rng.integers(0, 300, (2, B, S))

    def launched():
        enc.launch(True)
        return backend.core.download(enc.pooled, (B, cfg.d_model)), backend.core.download(enc.x, (B, S, cfg.d_model), enc.code)

    enc.set_inputs(ids, mask)
    want = launched()
    for earlier in (None, masks["right"][::-1].copy()):
        enc.forward(before, earlier)
        enc.forward(ids, mask)
        for _ in range(2):
            for got, w in zip(launched(), want):
                np.testing.assert_array_equal(got, w)
