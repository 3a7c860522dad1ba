"""Device-resident encoder forwards built from the hot-path kernels: the BERT-style post-LN encoder
(BertEncoder) and the pre-norm / rotary / GeGLU one (PreNormEncoder, further down).

Mirrors the forward recipe of the reference's VulkanSentenceTransformer
(utils/vulkan_sentence_transformer.py): embeddings = token + token-type 0 + position, then
LayerNorm (:563-747); per layer the post-LN block of _forward_layer (:972-1035) with the
Q/K/V projections fused into one packed weight; masked mean pooling and L2 normalisation
(:1177-1201).  Weights and activations live in HBM for the whole forward; only token ids and
the attention mask go in and the pooled embeddings (or the hidden states) come out.
"""
import ctypes
from dataclasses import dataclass

import numpy as np

from . import _lib as L
from .backend.core import HipCore, dtype_code


@dataclass
class EncoderConfig:
    layers: int = 12
    d_model: int = 768
    heads: int = 12
    d_ff: int = 3072
    vocab: int = 30522
    max_pos: int = 512
    eps: float = 1e-5          # the reference hard-codes 1e-5 in the layer LayerNorms (:1004, :1026)
    emb_eps: float = None      # embedding LayerNorm: the checkpoint's own eps in the reference (:729-736); None = eps

    @property
    def head_dim(self):
        return self.d_model // self.heads

    @property
    def embedding_eps(self):
        return self.eps if self.emb_eps is None else self.emb_eps


BERT_BASE = EncoderConfig()
MINILM_L6 = EncoderConfig(layers=6, d_model=384, heads=12, d_ff=1536)

_MATS = ("w_qkv", "w_o", "w_ff1", "w_ff2")
_VECS = ("b_qkv", "b_o", "ln1_g", "ln1_b", "b_ff1", "b_ff2", "ln2_g", "ln2_b")


def random_bert_weights(cfg, seed=0, std=0.02):
    """Random-init weights in the reference's (out_features, in_features) layout: matrices
    ~N(0,std), biases 0, LayerNorm gamma 1 / beta 0."""
    rng = np.random.default_rng(seed)
    d, ff = cfg.d_model, cfg.d_ff
    n = lambda *s: (rng.standard_normal(s) * std).astype(np.float32)
    w = {"tok_emb": n(cfg.vocab, d), "pos_emb": n(cfg.max_pos, d), "type_emb": n(2, d),
         "emb_ln_g": np.ones(d, np.float32), "emb_ln_b": np.zeros(d, np.float32), "layers": []}
    for _ in range(cfg.layers):
        w["layers"].append({
            "w_qkv": n(3 * d, d), "b_qkv": np.zeros(3 * d, np.float32),
            "w_o": n(d, d), "b_o": np.zeros(d, np.float32),
            "ln1_g": np.ones(d, np.float32), "ln1_b": np.zeros(d, np.float32),
            "w_ff1": n(ff, d), "b_ff1": np.zeros(ff, np.float32),
            "w_ff2": n(d, ff), "b_ff2": np.zeros(d, np.float32),
            "ln2_g": np.ones(d, np.float32), "ln2_b": np.zeros(d, np.float32)})
    return w


def _token_ids(input_ids):
    """ids as a contiguous int64 array, wrapped to 32 bits the way a cast to the kernels' int32 would"""
    ids = np.ascontiguousarray(input_ids)
    return ids if ids.dtype == np.int64 else ids.astype(np.int32, copy=False).astype(np.int64)


class _Slice:
    """a part of a device buffer"""
    __slots__ = ("ptr", "nbytes")

    def __init__(self, ptr, nbytes):
        self.ptr, self.nbytes = ptr, nbytes


class _Inputs:
    """Device memory for one batch's ids and mask, and behind them for the same batch without its padding: what forward()
    sends there in one transfer leaves launch() everything it reads."""
    __slots__ = ("buffer", "ids", "mask", "packed")

    def __init__(self, core, B, S):
        n = 4 * _Inputs.plane(B * S)
        self.buffer = core.alloc(2 * n + 4 * (B + 1 + 2 * B * S))
        self.ids, self.mask = _Slice(self.buffer.ptr, 4 * B * S), _Slice(self.buffer.ptr + n, 4 * B * S)
        self.packed = _Slice(self.buffer.ptr + 2 * n, 4 * (B + 1 + 2 * B * S))

    @staticmethod
    def plane(n):
        """values from the ids to the mask and from there to the packed batch: whole 256-byte units"""
        return (n + 63) // 64 * 64

    def free(self):
        self.buffer.free()


class _Packing:
    """What forward() makes of ids and mask in one native pass (grl_pack_inputs): both as the kernels take them, the real
    tokens' offsets, positions and ids, how many there are, and whether they form a batch without padding or one whose
    padding can be left out."""
    __slots__ = ("kind", "data", "packed", "B", "S", "rows", "longest")

    def __init__(self, lib, input_ids, attention_mask, vocab):
        ids = _token_ids(input_ids)
        if ids.ndim != 2:
            raise ValueError("input_ids must be (batch, seq_len)")
        B, S = ids.shape
        mask, kind = None, 0
        if attention_mask is not None:
            mask = np.asarray(attention_mask)
            mask = np.ascontiguousarray(mask, dtype=np.int64 if mask.dtype == np.int64 else np.float32)
            kind = 1 if mask.dtype == np.int64 else 2
            if mask.shape != (B, S):
                raise ValueError("attention_mask must be (batch, seq_len)")
        self.B, self.S = B, S
        plane = _Inputs.plane(B * S)
        self.data = np.empty(2 * plane + B + 1 + 2 * B * S, np.int32)
        self.packed = self.data[2 * plane:]
        rows, longest = ctypes.c_int64(), ctypes.c_int64()
        at = self.data.ctypes.data
        self.kind = lib.grl_pack_inputs(B, S, vocab, ids.ctypes.data, mask.ctypes.data if kind else None, kind, at, at + 4 * plane,
                                        at + 8 * plane, ctypes.byref(rows), ctypes.byref(longest))
        if self.kind == L.PACK_BAD_ID:
            raise IndexError("token id out of range")      # numpy indexing in the reference raises IndexError
        if self.kind < 0:
            L.check(self.kind, "pack_inputs")
        self.rows, self.longest = rows.value, longest.value

    @property
    def full(self):
        """no padding at all: a rectangular batch that needs no mask"""
        return self.kind == L.PACK_PREFIX and self.rows == self.B * self.S

    def upload_full(self, core, inputs):
        """the ids of a batch without padding (a mask of ones changes nothing)"""
        L.check(core.lib.grl_h2d(core.ctx, inputs.ids.ptr, self.data.ctypes.data, 4 * self.B * self.S), "upload ids")

    def upload(self, core, inputs):
        """ids, mask and offsets | positions | ids of the batch without its padding, in one transfer -> (ragged batch, device
        address of the latter ids)"""
        n = self.data.size - self.packed.size + self.B + 1 + 2 * self.rows
        L.check(core.lib.grl_h2d(core.ctx, inputs.ids.ptr, self.data.ctypes.data, n * 4), "upload batch")
        positions = inputs.packed.ptr + 4 * (self.B + 1)
        return L.Ragged(inputs.packed.ptr, positions, self.B, self.rows, self.longest), positions + 4 * self.rows


class BertEncoder:
    """forward(pool=True) leaves the padding of a batch out: the real tokens are stored back to back and every kernel sees
    those rows only (no result depends on a padded position: it is masked as a key and left out of the mean).  The batch
    keeps its rectangular form where hidden states come back (pool=False), where a mask holds other values than 0 and 1, and
    in bf16 where tokens are masked in front of or between kept ones.

    fused=None (default): both LayerNorms of every layer are folded into the GEMMs around them whenever the
    direct-to-LDS GEMM kernels take the layer's shapes (d_model and d_ff multiples of 64 in bf16, 32 in fp32) and the
    batch has at least FUSED_MIN_ROWS token rows (fp32: or FUSED_MIN_VALUES_F32 hidden values), or in bf16 few enough for the form without
    statistics passes: the residual stream then travels as raw rows plus row statistics and no LayerNorm pass runs over HBM between the embedding and the final LayerNorm
    (grl_bert_layers_fwd_fused).  Other batches run the seven-launch layer with its two LayerNorm passes (grl_bert_layer_fwd): a
    handful of token rows make a handful of tiles, the plain GEMMs then take tiles down to 32 x 32 while the fused layer's residual
    GEMM has none below 64 x 128, and the LayerNorm passes it saves cost next to nothing there.  Both weight
    sets stay resident.  fused=False always takes the seven-launch layer;
    fused=True always the fused one, and raises for shapes it does not take."""
    # us per forward, seven launches a layer -> fused: fp32 768 wide, 12 layers: 2048 rows 2856 -> 3048, 4096 rows level, 6400 rows
    # 7153 -> 6911; 384 wide, 6 layers: 4096 rows 942 -> 951, 6400 rows level; 128 wide, 4 layers, 20000 rows 453 -> 432.  In fp32 hidden
    # states are nearer to float64 with it (768 wide, 4400 rows: 7.35e-7 against 7.50e-7).  In bf16 they are not: the residual product's sum
    # is rounded before the residual is added, and the raw row once more in front of the last LayerNorm (twelve seeds each: 768 wide,
    # 2880 rows 8.86e-3 against 8.81e-3, 384 wide, 6400 rows 6.335e-3 against 6.327e-3).  So the bf16 line stands where the time saved is
    # more than a few per cent, not at the crossover (768 wide: 1536 rows 919 -> 884 us, 4096 rows 1473 -> 1403).
    FUSED_MIN_ROWS = 8192
    FUSED_MIN_VALUES_F32 = 3 << 20          # or, in fp32, so many values of the hidden states (rows x d_model)
    # bf16: up to so many values a layer runs as five launches without a LayerNorm pass (grl_bert_layer_fwd_rows): rows x the widest
    # activation (3 d_model or d_ff) up to the first, or rows x d_ff up to the second.  us per forward, seven launches -> five: d_ff 3072 /
    # 768 wide / 12 layers: 128 rows 517 -> 399, 320 rows 536 -> 449, 512 rows 642 -> 560, 640 rows 667 -> 584, 768 rows 732 -> 692;
    # 1536 / 384 / 6 layers: 256 rows 227 -> 196, 768 rows 267 -> 250, 1280 rows 294 -> 271, 1536 rows 331 -> 324.  Where d_ff is narrow the
    # QKV product is on far more 32 x 32 tiles than there are CUs (4 layers: 768 / 768 wide, 2560 rows 298 -> 336; 1536 / 768, 1500 rows
    # 293 -> 311; 256 / 256, 6000 rows 218 -> 253).  Hidden states are nearer to float64 than those of the seven launches (768 wide, 448 to 760
    # rows 0.975 of their error, 384 wide, 896 to 1500 rows 0.992 to 0.995).  In fp32 the two forms are within 4 % of each other from 128 rows on and the seven launches ahead below.
    ROWS_MAX_OUTPUTS, ROWS_MAX_FF = 9 << 18, 5 << 18

    def __init__(self, core, cfg, weights, dtype="fp32", fused=None):
        self.core = core.core if hasattr(core, "core") else core
        if not isinstance(self.core, HipCore):
            raise TypeError("BertEncoder needs a Compute() backend or its HipCore")
        if cfg.head_dim * cfg.heads != cfg.d_model:
            raise ValueError("d_model must be heads*head_dim")
        self.cfg, self.dtype, self.code = cfg, dtype, dtype_code(dtype)
        c = self.core
        self._keep = []                       # device buffers owned by the encoder
        up = lambda a, code=L.GRL_F32: self._own(c.upload(a, code))
        self.tok, self.pos, self.typ = up(weights["tok_emb"]), up(weights["pos_emb"]), up(weights["type_emb"])
        self.emb_g, self.emb_b = up(weights["emb_ln_g"]), up(weights["emb_ln_b"])
        self.layer_structs = []
        for lw in weights["layers"]:
            s = L.BertLayer()
            for k in _MATS:
                setattr(s, k, up(lw[k], self.code).ptr)
            for k in _VECS:
                setattr(s, k, up(np.asarray(lw[k]).reshape(-1)).ptr)
            self.layer_structs.append(s)
        slab = 64 if self.code == L.GRL_BF16 else 32
        eligible = cfg.d_model % slab == 0 and cfg.d_ff % slab == 0 and cfg.layers > 0
        if fused and not eligible:
            raise ValueError(f"the fused layer needs d_model and d_ff to be multiples of {slab} in {dtype}")
        self.fused = eligible if fused is None else bool(fused)
        self._fused_min_rows = self.fused_min_rows(cfg.d_model, self.code) if fused is None else 0
        few = fused is None and self.fused and self.code == L.GRL_BF16
        self._rows_max = self.rows_max(cfg.d_model, cfg.d_ff) if few else 0
        self.fused_structs = []
        if self.fused:
            # every GEMM that reads a LayerNorm's output gets that norm folded into its weight (once, here):
            # QKV of layer l reads the embedding norm (l = 0) or the second norm of layer l-1, FFN1 reads ln1
            d, ff = cfg.d_model, cfg.d_ff
            es = 2 if self.code == L.GRL_BF16 else 4

            def fold(w, b_ptr, g_ptr, bt_ptr, n, k):
                raw = c.upload(w)
                ws, cs, bf = self._own(c.alloc(n * k * es)), self._own(c.alloc(n * 4)), self._own(c.alloc(n * 4))
                L.check(c.lib.grl_ln_fold_f32(c.ctx, self.code, n, k, raw.ptr, g_ptr, bt_ptr, b_ptr, ws.ptr, cs.ptr, bf.ptr), "fold layernorm")
                raw.free()
                return ws.ptr, cs.ptr, bf.ptr
            in_g, in_b = self.emb_g.ptr, self.emb_b.ptr
            for s, lw in zip(self.layer_structs, weights["layers"]):
                f = L.BertLayerFused()
                f.ws_qkv, f.c_qkv, f.bf_qkv = fold(lw["w_qkv"], s.b_qkv, in_g, in_b, 3 * d, d)
                f.in_g, f.in_b = in_g, in_b
                f.w_o, f.b_o, f.ln1_g, f.ln1_b = s.w_o, s.b_o, s.ln1_g, s.ln1_b
                f.ws_ff1, f.c_ff1, f.bf_ff1 = fold(lw["w_ff1"], s.b_ff1, s.ln1_g, s.ln1_b, ff, d)
                f.w_ff2, f.b_ff2 = s.w_ff2, s.b_ff2
                self.fused_structs.append(f)
                in_g, in_b = s.ln2_g, s.ln2_b
            self._fused_array = (L.BertLayerFused * len(self.fused_structs))(*self.fused_structs)
        self._shape = None

    @classmethod
    def fused_min_rows(cls, d_model, code):
        """token rows from which a batch runs the fused layers by default"""
        return cls.FUSED_MIN_ROWS if code == L.GRL_BF16 else min(cls.FUSED_MIN_ROWS, -(-cls.FUSED_MIN_VALUES_F32 // d_model))

    @classmethod
    def rows_max(cls, d_model, d_ff):
        """token rows up to which a bf16 batch runs the five-launch layers by default"""
        return max(cls.ROWS_MAX_OUTPUTS // max(3 * d_model, d_ff), cls.ROWS_MAX_FF // d_ff)

    def _own(self, buf):
        self._keep.append(buf)
        return buf

    # ---- device-side state for one (B,S): hidden states, workspace, ids, mask, pooled output
    def prepare(self, B, S):
        if self._shape == (B, S):
            return
        self.release_activations()
        cfg, c = self.cfg, self.core
        if S > cfg.max_pos:
            raise ValueError(f"sequence length {S} exceeds max_pos {cfg.max_pos}")
        es = 2 if self.code == L.GRL_BF16 else 4
        self.fused_now = self.fused and B * S >= self._fused_min_rows        # which layer form this batch runs
        ws = c.lib.grl_bert_layer_workspace(self.code, B, S, cfg.heads, cfg.head_dim, cfg.d_ff)
        if self.fused:                       # without its padding the batch may run any form
            ws = max(ws, c.lib.grl_bert_layers_fused_workspace(self.code, B, S, cfg.heads, cfg.head_dim, cfg.d_ff))
        self.x = c.alloc(B * S * cfg.d_model * es)
        self.stats = c.alloc(max(B * S, 1) * 8)        # {1/sd, mean/sd} per row of the raw residual stream (fused layers)
        self.ws = c.alloc(ws)
        self.inputs = _Inputs(c, B, S)
        self.ids, self.mask = self.inputs.ids, self.inputs.mask
        self.pooled = c.alloc(B * cfg.d_model * 4)
        self._shape = (B, S)

    def release_activations(self):
        if self._shape is not None:
            for b in (self.x, self.stats, self.ws, self.inputs, self.pooled):
                b.free()
            self._shape = None

    def set_inputs(self, input_ids, attention_mask=None):
        ids = np.ascontiguousarray(input_ids, dtype=np.int32)
        if ids.ndim != 2:
            raise ValueError("input_ids must be (batch, seq_len)")
        if ids.size and (ids.min() < 0 or ids.max() >= self.cfg.vocab):
            raise IndexError("token id out of range")      # numpy indexing in the reference raises IndexError
        B, S = ids.shape
        self.prepare(B, S)
        c = self.core
        L.check(c.lib.grl_h2d(c.ctx, self.ids.ptr, ids.ctypes.data, ids.nbytes), "upload ids")
        self.has_mask = attention_mask is not None
        if self.has_mask:
            m = np.ascontiguousarray(attention_mask, dtype=np.float32)
            if m.shape != (B, S):
                raise ValueError("attention_mask must be (batch, seq_len)")
            L.check(c.lib.grl_h2d(c.ctx, self.mask.ptr, m.ctypes.data, m.nbytes), "upload mask")

    def _set_full(self, p):
        """set_inputs for a batch without padding"""
        self.prepare(p.B, p.S)
        p.upload_full(self.core, self.inputs)
        self.has_mask = False

    def _set_packed(self, p):
        """set_inputs for a batch that runs without its padding -> what upload() returns"""
        self.prepare(p.B, p.S)
        self.has_mask = True
        return p.upload(self.core, self.inputs)

    def launch(self, pool=True):
        """Enqueue one full forward of the batch that set_inputs() or forward() had last, in its rectangular form, on the
        context stream (no host synchronisation); its hidden states are left in x as (B, S, d)."""
        B, S = self._shape
        cfg, c, lib = self.cfg, self.core, self.core.lib
        mask = self.mask.ptr if self.has_mask else None
        if 0 < B * S <= self._rows_max:
            L.check(lib.grl_embed(c.ctx, self.code, B, S, cfg.d_model, cfg.vocab, self.ids.ptr, self.tok.ptr, self.pos.ptr,
                                  self.typ.ptr, self.x.ptr), "embedding")
            in_eps = cfg.embedding_eps
            for f in self.fused_structs:
                L.check(lib.grl_bert_layer_fwd_rows(c.ctx, self.code, B, S, cfg.heads, cfg.head_dim, cfg.d_ff, ctypes.byref(f), mask,
                                                    in_eps, cfg.eps, self.x.ptr, self.ws.ptr), "bert_layer_fwd_rows")
                in_eps = cfg.eps
            self._last_layernorm(B * S)
        elif self.fused_now and B * S > 0:
            # raw embedding rows + their statistics; the layers pass raw rows and row statistics on; the last layer's second
            # LayerNorm is the one pass that writes normalised rows
            L.check(lib.grl_embed(c.ctx, self.code, B, S, cfg.d_model, cfg.vocab, self.ids.ptr, self.tok.ptr, self.pos.ptr,
                                  self.typ.ptr, self.x.ptr), "embedding")
            L.check(lib.grl_ln_stats(c.ctx, self.code, B * S, cfg.d_model, self.x.ptr, cfg.embedding_eps, self.stats.ptr), "embedding statistics")
            L.check(lib.grl_bert_layers_fwd_fused(c.ctx, self.code, B, S, cfg.heads, cfg.head_dim, cfg.d_ff, self._fused_array, cfg.layers,
                                                  mask, cfg.eps, self.x.ptr, self.stats.ptr, self.ws.ptr), "bert_layers_fwd_fused")
            self._last_layernorm(B * S)
        else:
            L.check(lib.grl_embed_layernorm(c.ctx, self.code, B, S, cfg.d_model, cfg.vocab, self.ids.ptr, self.tok.ptr,
                                            self.pos.ptr, self.typ.ptr, self.emb_g.ptr, self.emb_b.ptr, cfg.embedding_eps,
                                            self.x.ptr), "embedding + layernorm")
            for s in self.layer_structs:
                L.check(lib.grl_bert_layer_fwd(c.ctx, self.code, B, S, cfg.heads, cfg.head_dim, cfg.d_ff, ctypes.byref(s),
                                               mask, cfg.eps, self.x.ptr, self.ws.ptr), "bert_layer_fwd")
        if pool:
            L.check(lib.grl_mean_pool(c.ctx, self.code, B, S, cfg.d_model, self.x.ptr, mask, self.pooled.ptr, 1), "mean_pool")

    def _last_layernorm(self, rows):
        """raw rows -> the last layer's normalised ones"""
        c, last = self.core, self.layer_structs[-1]
        L.check(c.lib.grl_layernorm(c.ctx, self.code, rows, self.cfg.d_model, self.x.ptr, None, last.ln2_g, last.ln2_b, self.cfg.eps,
                                    self.x.ptr), "final layernorm")

    def _launch_packed(self, rg, ids):
        """launch() on the batch without its padding, always pooled"""
        cfg, c, lib = self.cfg, self.core, self.core.lib
        r = ctypes.byref(rg)
        if 0 < rg.rows <= self._rows_max:
            L.check(lib.grl_embed_ragged(c.ctx, self.code, r, cfg.d_model, cfg.vocab, ids, self.tok.ptr, self.pos.ptr, self.typ.ptr,
                                         self.x.ptr), "embedding")
            in_eps = cfg.embedding_eps
            for f in self.fused_structs:
                L.check(lib.grl_bert_layer_fwd_rows_ragged(c.ctx, self.code, r, cfg.heads, cfg.head_dim, cfg.d_ff, ctypes.byref(f), in_eps,
                                                           cfg.eps, self.x.ptr, self.ws.ptr), "bert_layer_fwd_rows")
                in_eps = cfg.eps
            self._last_layernorm(rg.rows)
        elif self.fused and rg.rows >= self._fused_min_rows and rg.rows > 0:
            L.check(lib.grl_embed_ragged(c.ctx, self.code, r, cfg.d_model, cfg.vocab, ids, self.tok.ptr, self.pos.ptr, self.typ.ptr,
                                         self.x.ptr), "embedding")
            L.check(lib.grl_ln_stats(c.ctx, self.code, rg.rows, cfg.d_model, self.x.ptr, cfg.embedding_eps, self.stats.ptr), "embedding statistics")
            L.check(lib.grl_bert_layers_fwd_fused_ragged(c.ctx, self.code, r, cfg.heads, cfg.head_dim, cfg.d_ff, self._fused_array, cfg.layers,
                                                         cfg.eps, self.x.ptr, self.stats.ptr, self.ws.ptr), "bert_layers_fwd_fused")
            self._last_layernorm(rg.rows)
        else:
            L.check(lib.grl_embed_layernorm_ragged(c.ctx, self.code, r, cfg.d_model, cfg.vocab, ids, self.tok.ptr, self.pos.ptr, self.typ.ptr,
                                                   self.emb_g.ptr, self.emb_b.ptr, cfg.embedding_eps, self.x.ptr), "embedding + layernorm")
            for s in self.layer_structs:
                L.check(lib.grl_bert_layer_fwd_ragged(c.ctx, self.code, r, cfg.heads, cfg.head_dim, cfg.d_ff, ctypes.byref(s), cfg.eps,
                                                      self.x.ptr, self.ws.ptr), "bert_layer_fwd")
        L.check(lib.grl_mean_pool_ragged(c.ctx, self.code, r, cfg.d_model, self.x.ptr, 0, self.pooled.ptr, 1), "mean_pool")

    def forward(self, input_ids, attention_mask=None, pool=True):
        """pool=True -> L2-normalised mean-pooled embeddings (B, d); False -> hidden states (B,S,d)."""
        p = _Packing(self.core.lib, input_ids, attention_mask, self.cfg.vocab)
        # Padding on the right leaves every key in the attention tile it has in the rectangular batch, so pooled embeddings
        # agree with the mean of pool=False's hidden states to the last bits.  Tokens kept elsewhere move to other tiles,
        # where bf16 rounds the softmax weights against another reference (1e-3 measured): fp32 only.
        packs = p.kind == L.PACK_PREFIX or (p.kind == L.PACK_SCATTERED and self.code == L.GRL_F32)
        if pool and packs and not p.full and self.cfg.head_dim <= 128:
            self._launch_packed(*self._set_packed(p))
        else:
            if p.full:
                self._set_full(p)
            else:
                self.set_inputs(input_ids, attention_mask)
            self.launch(pool)
        B, S = self._shape
        if pool:
            return self.core.download(self.pooled, (B, self.cfg.d_model))
        return self.core.download(self.x, (B, S, self.cfg.d_model), self.code)

    def flops_per_forward(self, B, S):
        """2*M*N*K per GEMM + 4*B*H*S^2*D for attention (dense count)."""
        cfg = self.cfg
        M, d, ff = B * S, cfg.d_model, cfg.d_ff
        per_layer = 2 * M * d * 3 * d + 2 * M * d * d + 2 * 2 * M * d * ff + 4 * B * cfg.heads * S * S * cfg.head_dim
        return cfg.layers * per_layer


# ------------------------------------------------------------------------------------------------
@dataclass
class PreNormEncoderConfig:
    """ModernBERT-shaped encoder: token embeddings only, rotary positions, GeGLU MLP."""
    layers: int = 22
    d_model: int = 768
    heads: int = 12
    d_ff: int = 1152           # width of each GeGLU half (Wi is (2*d_ff, d_model))
    vocab: int = 50368
    eps: float = 1e-5          # the reference hard-codes 1e-5 for the layer norm in front of the MLP (:901)
    emb_eps: float = 1e-5
    final_eps: float = 1e-5
    rope_base: float = 10000.0
    rope_scaling: float = 1.0

    @property
    def head_dim(self):
        return self.d_model // self.heads


def random_prenorm_weights(cfg, seed=0, std=0.02):
    """Random-init weights, (out_features, in_features) matrices ~N(0,std), biases 0, norms 1 / 0."""
    rng = np.random.default_rng(seed)
    d, ff = cfg.d_model, cfg.d_ff
    n = lambda *s: (rng.standard_normal(s) * std).astype(np.float32)
    one, zero = (lambda k: np.ones(k, np.float32)), (lambda k: np.zeros(k, np.float32))
    w = {"tok_emb": n(cfg.vocab, d), "emb_ln_g": one(d), "emb_ln_b": zero(d),
         "final_ln_g": one(d), "final_ln_b": zero(d), "layers": []}
    for _ in range(cfg.layers):
        w["layers"].append({
            "w_qkv": n(3 * d, d), "b_qkv": zero(3 * d), "w_o": n(d, d), "b_o": zero(d),
            "ffn_ln_g": one(d), "ffn_ln_b": zero(d),
            "w_ff_in": n(ff, d), "b_ff_in": zero(ff), "w_ff_gate": n(ff, d), "b_ff_gate": zero(ff),
            "w_ff2": n(d, ff), "b_ff2": zero(d)})
    return w


class PreNormEncoder:
    """Device-resident forward of the reference's pre-norm branch
    (utils/vulkan_sentence_transformer.py:799-970 per layer; encode :1146-1183 around it):

        x = LN(tok_emb[ids]; emb)                                              (:1153-1155, :749-785)
        per layer:  x += Wo.Attn(rope(Wq x), rope(Wk x), Wv x; key mask)       (:806-893, no norm in front)
                    x += W2.(gelu(Wi_in.LN(x)) * (Wi_gate.LN(x)))              (:901-945)
        x = LN(x; final)   (only if final_ln_g is given, :1166-1175)
        pooled = x[:, 0, :] (first token), L2-normalised                       (:1179-1183, :1194-1201)

    Built from the same entry points as the post-LN encoder: the projection GEMMs, attention with the
    rotate-half rotation fused, the dual GEMM with the GELU gate, and the GEMM that adds the residual stream in
    place.  The LayerNorm in front of the MLP is folded into that dual GEMM (gamma into the two weights, beta into
    the biases, once at construction; the GEMM reads the residual stream itself and applies each row's mean and
    1/sd in its epilogue), so the normalised rows are never written.
    The packed Wqkv is one GEMM; attention reads its three column blocks in place.  The +-50 / +-1e6 clips the
    reference puts around the gate (:924-930) are not applied: they only act beyond those magnitudes."""

    def __init__(self, core, cfg, weights, dtype="fp32", stats_from_gemm=None):
        self.core = core.core if hasattr(core, "core") else core
        if not isinstance(self.core, HipCore):
            raise TypeError("PreNormEncoder needs a Compute() backend or its HipCore")
        self._stats_from_gemm = stats_from_gemm        # None: wherever the kernel takes the width
        # Few rows (rows x d_ff up to this): the gated GEMM takes the statistics of its rows itself.  us per forward of 22 layers,
        # 768 wide, d_ff 1152: bf16 128 rows 796 -> 637, 640 rows 1117 -> 896, 896 rows 1164 -> 972; fp32 20 rows 1630 -> 1084,
        # 896 rows 3327 -> 2829, 1280 rows 3915 -> 3744, 2048 rows 5629 -> 5651
        half = dtype_code(dtype) == L.GRL_BF16
        takes = cfg.d_model % (64 if half else 32) == 0 and cfg.d_ff % 4 == 0
        self._own_max = (1 << 20 if half else 7 << 18) if stats_from_gemm is None and takes else 0
        if cfg.head_dim * cfg.heads != cfg.d_model or cfg.head_dim % 2 or cfg.head_dim > 128:
            raise ValueError("d_model must be heads*head_dim with an even head_dim up to 128 (rotary positions)")
        self.cfg, self.dtype, self.code = cfg, dtype, dtype_code(dtype)
        c = self.core
        self._keep = []
        up = lambda a, code=L.GRL_F32: self._own(c.upload(a, code))
        vec = lambda a: up(np.asarray(a, np.float32).reshape(-1))
        self.tok = up(weights["tok_emb"])
        self.emb_g, self.emb_b = vec(weights["emb_ln_g"]), vec(weights["emb_ln_b"])
        self.final = None
        if weights.get("final_ln_g") is not None:
            self.final = (vec(weights["final_ln_g"]), vec(weights["final_ln_b"]))
        self.layers = []
        es = 2 if self.code == L.GRL_BF16 else 4
        d, ff = cfg.d_model, cfg.d_ff
        for lw in weights["layers"]:
            entry = {k: up(lw[k], self.code) for k in ("w_qkv", "w_o", "w_ff2")}
            entry.update({k: vec(lw[k]) for k in ("b_qkv", "b_o", "b_ff2")})
            g, bt = c.upload(np.asarray(lw["ffn_ln_g"], np.float32).reshape(-1)), c.upload(np.asarray(lw["ffn_ln_b"], np.float32).reshape(-1))
            for name in ("gate", "in"):
                raw = c.upload(lw["w_ff_" + name])
                b = c.upload(np.asarray(lw["b_ff_" + name], np.float32).reshape(-1))
                ws, cs, bf = self._own(c.alloc(ff * d * es)), self._own(c.alloc(ff * 4)), self._own(c.alloc(ff * 4))
                L.check(c.lib.grl_ln_fold_f32(c.ctx, self.code, ff, d, raw.ptr, g.ptr, bt.ptr, b.ptr, ws.ptr, cs.ptr, bf.ptr), "fold mlp layernorm")
                entry["ws_" + name], entry["cs_" + name], entry["bf_" + name] = ws, cs, bf
                raw.free(); b.free()
            g.free(); bt.free()
            self.layers.append(entry)
        self._shape = None

    def _own(self, buf):
        self._keep.append(buf)
        return buf

    def prepare(self, B, S):
        if self._shape == (B, S):
            return
        self.release_activations()
        cfg, c = self.cfg, self.core
        es = 2 if self.code == L.GRL_BF16 else 4
        act = B * S * cfg.d_model * es
        self.x, self.att = (c.alloc(act) for _ in range(2))
        self.stats = c.alloc(B * S * 8)                # {1/sd, mean/sd} per row, for the GEMM that carries the MLP's LayerNorm
        # The row statistics come out of the epilogue of the output projection that writes the rows (the GEMM entry point
        # that adds LayerNorm(residual) and reduces the moments of what it stores, here with the identity in place of the
        # LayerNorm: statistics {1, 0}, scale 1, shift 0) where that kernel takes the shape; else from a pass over the rows.
        slab = 64 if self.code == L.GRL_BF16 else 32
        self.stats_from_gemm = cfg.d_model % slab == 0 if self._stats_from_gemm is None else bool(self._stats_from_gemm)
        if self.stats_from_gemm and cfg.d_model % slab:
            raise ValueError(f"row statistics out of the GEMM epilogue need d_model to be a multiple of {slab}")
        if self.stats_from_gemm:
            ident = np.zeros((B * S, 2), np.float32)
            ident[:, 0] = 1.0
            self.ident_stats = c.upload_raw(ident)
            self.ones, self.zeros = c.upload_raw(np.ones(cfg.d_model, np.float32)), c.upload_raw(np.zeros(cfg.d_model, np.float32))
            self.part = c.alloc(int(c.lib.grl_gemm_nt_resln_workspace(B * S, cfg.d_model)))
        self.qkv = c.alloc(3 * act)                    # packed (M, 3d): Q, K, V are its three column blocks
        self.h = c.alloc(B * S * cfg.d_ff * es)
        self.inputs = _Inputs(c, B, S)
        self.ids, self.mask = self.inputs.ids, self.inputs.mask
        first = np.zeros((B, S), np.float32)
        first[:, 0] = 1.0                              # "mean" over the first token only = that token
        self.first = c.upload_raw(first)
        self.pooled = c.alloc(B * cfg.d_model * 4)
        self._shape = (B, S)

    def release_activations(self):
        if self._shape is not None:
            for b in (self.x, self.qkv, self.att, self.stats, self.h, self.inputs, self.first, self.pooled):
                b.free()
            if self.stats_from_gemm:
                for b in (self.ident_stats, self.ones, self.zeros, self.part):
                    b.free()
            self._shape = None

    def set_inputs(self, input_ids, attention_mask=None):
        ids = np.ascontiguousarray(input_ids, dtype=np.int32)
        if ids.ndim != 2 or ids.shape[1] == 0:
            raise ValueError("input_ids must be (batch, seq_len) with seq_len > 0")
        if ids.size and (ids.min() < 0 or ids.max() >= self.cfg.vocab):
            raise IndexError("token id out of range")
        B, S = ids.shape
        self.prepare(B, S)
        c = self.core
        L.check(c.lib.grl_h2d(c.ctx, self.ids.ptr, ids.ctypes.data, ids.nbytes), "upload ids")
        self.has_mask = attention_mask is not None
        if self.has_mask:
            m = np.ascontiguousarray(attention_mask, dtype=np.float32)
            if m.shape != (B, S):
                raise ValueError("attention_mask must be (batch, seq_len)")
            L.check(c.lib.grl_h2d(c.ctx, self.mask.ptr, m.ctypes.data, m.nbytes), "upload mask")

    _set_full, _set_packed = BertEncoder._set_full, BertEncoder._set_packed

    def launch(self, pool=True):
        """Enqueue one full forward of the batch that set_inputs() or forward() had last (as in BertEncoder)."""
        self._launch(pool, None, self.ids.ptr)

    def _launch(self, pool, rg, ids):
        """rg: the batch without its padding (pool is then True), or None for the rectangular one"""
        B, S = self._shape
        cfg, c, lib, code = self.cfg, self.core, self.core.lib, self.code
        M, d, ff, H, D = B * S if rg is None else rg.rows, cfg.d_model, cfg.d_ff, cfg.heads, cfg.head_dim
        own_stats = 0 < M * ff <= self._own_max
        if rg is None:
            mask = self.mask.ptr if self.has_mask else None
            L.check(lib.grl_embed_layernorm(c.ctx, code, B, S, d, cfg.vocab, ids, self.tok.ptr, None, None,
                                            self.emb_g.ptr, self.emb_b.ptr, cfg.emb_eps, self.x.ptr), "embedding + layernorm")
        else:
            L.check(lib.grl_embed_layernorm_ragged(c.ctx, code, ctypes.byref(rg), d, cfg.vocab, ids, self.tok.ptr, None, None,
                                                   self.emb_g.ptr, self.emb_b.ptr, cfg.emb_eps, self.x.ptr), "embedding + layernorm")
        for w in self.layers:
            # one GEMM with the packed weight, rotating queries and keys on its way out where its kernel can; attention reads Q, K, V
            # as column blocks of its output
            L.check(lib.grl_rotary_attention(c.ctx, code, B, S, None if rg is None else ctypes.byref(rg), H, D, self.x.ptr, w["w_qkv"].ptr,
                                             w["b_qkv"].ptr, mask if rg is None else None, self.qkv.ptr, self.att.ptr, cfg.rope_base,
                                             cfg.rope_scaling), "q/k/v projection, attention")
            # LayerNorm + dual GEMM; the dual GEMM activates its second ("up") operand: that is the first half of Wi here
            if own_stats:
                L.check(lib.grl_gemm_nt_res(c.ctx, code, code, M, d, d, self.att.ptr, w["w_o"].ptr, w["b_o"].ptr, self.x.ptr,
                                            self.x.ptr), "output projection + residual")
                L.check(lib.grl_ln_glu_nt_rows(c.ctx, code, M, ff, d, self.x.ptr, w["ws_gate"].ptr, w["ws_in"].ptr, w["cs_gate"].ptr,
                                               w["cs_in"].ptr, w["bf_gate"].ptr, w["bf_in"].ptr, cfg.eps, self.h.ptr, L.EPI_GELU),
                        "mlp layernorm + geglu")
            elif self.stats_from_gemm:
                L.check(lib.grl_resln_ln_glu(c.ctx, code, M, d, d, ff, self.att.ptr, w["w_o"].ptr, w["b_o"].ptr, self.x.ptr,
                                             self.ident_stats.ptr, self.ones.ptr, self.zeros.ptr, self.x.ptr, w["ws_gate"].ptr, w["ws_in"].ptr,
                                             w["cs_gate"].ptr, w["cs_in"].ptr, w["bf_gate"].ptr, w["bf_in"].ptr, cfg.eps, self.stats.ptr,
                                             self.part.ptr, self.h.ptr, L.EPI_GELU), "output projection + residual, mlp layernorm + geglu")
            else:
                L.check(lib.grl_gemm_nt_res(c.ctx, code, code, M, d, d, self.att.ptr, w["w_o"].ptr, w["b_o"].ptr, self.x.ptr,
                                            self.x.ptr), "output projection + residual")
                L.check(lib.grl_ln_glu_nt(c.ctx, code, code, M, ff, d, self.x.ptr, w["ws_gate"].ptr, w["ws_in"].ptr,
                                          w["cs_gate"].ptr, w["cs_in"].ptr, w["bf_gate"].ptr, w["bf_in"].ptr, cfg.eps,
                                          self.stats.ptr, self.h.ptr, L.EPI_GELU), "mlp layernorm + geglu")
            L.check(lib.grl_gemm_nt_res(c.ctx, code, code, M, d, ff, self.h.ptr, w["w_ff2"].ptr, w["b_ff2"].ptr, self.x.ptr,
                                        self.x.ptr), "mlp output + residual")
        if self.final is not None:
            L.check(lib.grl_layernorm(c.ctx, code, M, d, self.x.ptr, None, self.final[0].ptr, self.final[1].ptr,
                                      cfg.final_eps, self.x.ptr), "final layernorm")
        if rg is not None:
            L.check(lib.grl_mean_pool_ragged(c.ctx, code, ctypes.byref(rg), d, self.x.ptr, 1, self.pooled.ptr, 1), "first-token pool")
        elif pool:
            L.check(lib.grl_mean_pool(c.ctx, code, B, S, d, self.x.ptr, self.first.ptr, self.pooled.ptr, 1), "first-token pool")

    def forward(self, input_ids, attention_mask=None, pool=True):
        """pool=True -> L2-normalised first-token embeddings (B, d); False -> hidden states (B,S,d).  Pooled batches padded
        on the right run without their padding, as in BertEncoder (the first token has to be a real one)."""
        p = _Packing(self.core.lib, input_ids, attention_mask, self.cfg.vocab)
        if pool and not p.full and p.kind == L.PACK_PREFIX and (p.packed[1:p.B + 1] > p.packed[:p.B]).all():
            self._launch(True, *self._set_packed(p))
        else:
            if p.full and p.S > 0:
                self._set_full(p)
            else:
                self.set_inputs(input_ids, attention_mask)
            self.launch(pool)
        B, S = self._shape
        if pool:
            return self.core.download(self.pooled, (B, self.cfg.d_model))
        return self.core.download(self.x, (B, S, self.cfg.d_model), self.code)
