"""The work that is timed: calls a program makes through this package's public entry points.

Five families, each over the range of sizes it is used in:

  fnn        `backend.fnn.linear / fused_linear_gelu / fused_swiglu`, numpy in, numpy out (the operators of the README)
  attention  `backend.attention.flash_attention2(_rope)`, numpy in, numpy out
  encoder    `BertEncoder.forward` / `PreNormEncoder.forward`: token ids and attention mask in, sentence embeddings or
             hidden states out, weights resident
  mlp        the gated MLP on device-resident activations through the C interface: grl_swiglu_nt, then grl_gemm_nt
  device_attention  grl_fa2_fwd on device-resident Q, K, V

A case is a dict of plain values; `listed()` names twelve, `draw()` picks more of the same ranges.
"""
import functools
import math

import numpy as np
import torch

import grilly_amd
from grilly_amd import _lib as L
from grilly_amd.backend.core import dtype_code

# name -> (layers, d_model, heads, d_ff, vocab): the encoder shapes of the benchmark
ARCHS = {"bert_base": (12, 768, 12, 3072, 30522), "minilm_l6": (6, 384, 12, 1536, 30522), "prenorm": (22, 768, 12, 1152, 50368)}


def listed():
    return [
        # the README's first call: one small fp32 linear, where the call itself is the cost
        {"name": "linear_small", "family": "fnn", "op": "linear", "m": 32, "k": 384, "n": 128, "dtype": "fp32"},
        # the first half of a feed-forward block over a batch of token rows, called from numpy
        {"name": "linear_gelu_rows", "family": "fnn", "op": "fused_linear_gelu", "m": 4000, "k": 768, "n": 3072, "dtype": "fp32"},
        # the README's attention call: many short heads, numpy in and out
        {"name": "attention_small", "family": "attention", "b": 32, "s": 64, "h": 8, "d": 64, "causal": False, "rope": False, "dtype": "fp32"},
        # embedding one query while somebody waits for it
        {"name": "one_sentence_bf16", "family": "encoder", "arch": "bert_base", "dtype": "bf16", "b": 1, "s": 128, "pad": False, "pool": True},
        # a handful of sentences of unequal length in full precision
        {"name": "few_sentences_fp32", "family": "encoder", "arch": "bert_base", "dtype": "fp32", "b": 8, "s": 100, "pad": True, "pool": True},
        # bulk sentence embedding with the small model, padded batch, full precision
        {"name": "minilm_batch_fp32", "family": "encoder", "arch": "minilm_l6", "dtype": "fp32", "b": 64, "s": 256, "pad": True, "pool": True},
        # token features of a padded batch: the hidden states themselves come back
        {"name": "token_states_bf16", "family": "encoder", "arch": "minilm_l6", "dtype": "bf16", "b": 32, "s": 200, "pad": True, "pool": False},
        # bulk document embedding, every sequence cut to the model's length: the benchmark's headline
        {"name": "bert_full_bf16", "family": "encoder", "arch": "bert_base", "dtype": "bf16", "b": 128, "s": 512, "pad": False, "pool": True},
        # bulk embedding of texts as they come, padded to the longest
        {"name": "bert_padded_bf16", "family": "encoder", "arch": "bert_base", "dtype": "bf16", "b": 48, "s": 384, "pad": True, "pool": True},
        # the rotary, pre-norm encoder on a padded batch
        {"name": "prenorm_padded_bf16", "family": "encoder", "arch": "prenorm", "dtype": "bf16", "b": 32, "s": 300, "pad": True, "pool": True},
        # the large gated MLP of a language model's prefill
        {"name": "swiglu_mlp_bf16", "family": "mlp", "m": 16384, "k": 4096, "n": 11008, "dtype": "bf16"},
        # long causal attention with rotary positions
        {"name": "rope_attention_long", "family": "device_attention", "b": 4, "s": 8192, "h": 32, "d": 128, "causal": True, "rope": True, "dtype": "bf16"},
    ]


# ---------------------------------------------------------------------------------------------- drawn cases
MOST_FLOPS = 12.0e12            # bf16; an fp32 case counts sixteen times (the ratio of the two matrix rates)
MOST_HOST_BYTES = 72.0e6        # numpy arrays in and out of one call


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _near(rng, lo, hi, step, odd):
    """A size between lo and hi, spread over its logarithm: a multiple of `step`, or with probability `odd` any number."""
    v = _log(rng, lo, hi)
    return v if rng.random() < odd else max(step, v // step * step)


def _draw_one(rng):
    family = rng.choice(["fnn", "attention", "encoder", "encoder", "encoder", "mlp", "device_attention"])
    dtype = rng.choice(["fp32", "bf16"])
    if family == "fnn":
        return {"family": family, "op": rng.choice(["linear", "fused_linear_gelu", "fused_swiglu"]), "m": _log(rng, 1, 4000),
                "k": _near(rng, 64, 1024, 8, 0.2), "n": _near(rng, 64, 3072, 8, 0.2), "dtype": dtype}
    if family == "attention":
        return {"family": family, "b": _log(rng, 1, 32), "s": _log(rng, 16, 512), "h": rng.choice([4, 8, 12, 16]), "d": rng.choice([32, 64, 128]),
                "causal": rng.random() < 0.5, "rope": rng.random() < 0.5, "dtype": dtype}
    if family == "encoder":
        return {"family": family, "arch": rng.choice(sorted(ARCHS)), "dtype": dtype, "b": _log(rng, 1, 128), "s": _log(rng, 8, 512),
                "pad": rng.random() < 0.7, "pool": rng.random() < 0.8}
    if family == "mlp":
        return {"family": family, "m": _log(rng, 1, 16384), "k": _near(rng, 512, 4096, 64, 0.0), "n": _near(rng, 512, 11008, 64, 0.0), "dtype": dtype}
    return {"family": family, "b": _log(rng, 1, 32), "s": _log(rng, 128, 8192), "h": rng.choice([8, 12, 16, 32]), "d": rng.choice([32, 64, 128]),
            "causal": rng.random() < 0.5, "rope": rng.random() < 0.5, "dtype": dtype}


def draw(rng):
    while True:
        case = _draw_one(rng)
        w = work(case)
        host = w["bytes"] if case["family"] in ("fnn", "attention") else 0
        resident = 4.0 * case["b"] * case["s"] * case["h"] * case["d"] * _es(case) if case["family"] == "device_attention" else 0
        if w["flops"] * (16 if case["dtype"] == "fp32" else 1) <= MOST_FLOPS and host <= MOST_HOST_BYTES and resident <= 1.1e9:
            return case


# ---------------------------------------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=1)
def _backend():
    """One backend for the whole program, as its users keep it."""
    return grilly_amd.Compute(0)


def _es(case):
    return 2 if case["dtype"] == "bf16" else 4


def _normals(seed):
    """fp32 N(0, std) values from the seed, made on the GPU (numpy arrays where the call takes numpy)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return lambda shape, std=1.0: torch.randn(*shape, generator=gen, device="cuda") * std


def _padded_lengths(rng, case):
    """Sequence lengths of a batch padded to its longest: uniform in [s/8, s], one sequence of full length."""
    b, s = case["b"], case["s"]
    n = rng.integers(max(1, s // 8), s + 1, b)
    n[rng.integers(b)] = s
    return n


def _encoder(case, seed):
    layers, d, heads, ff, vocab = ARCHS[case["arch"]]
    normal = _normals(seed)
    mat = lambda *shape: normal(shape, 0.02).cpu().numpy()
    vec = lambda n, at: normal((n,), 0.02).add(at).cpu().numpy()
    w = {"tok_emb": mat(vocab, d), "emb_ln_g": vec(d, 1.0), "emb_ln_b": vec(d, 0.0), "layers": []}
    if case["arch"] == "prenorm":
        w.update(final_ln_g=vec(d, 1.0), final_ln_b=vec(d, 0.0))
        for _ in range(layers):
            w["layers"].append({"w_qkv": mat(3 * d, d), "b_qkv": vec(3 * d, 0.0), "w_o": mat(d, d), "b_o": vec(d, 0.0), "ffn_ln_g": vec(d, 1.0),
                                "ffn_ln_b": vec(d, 0.0), "w_ff_in": mat(ff, d), "b_ff_in": vec(ff, 0.0), "w_ff_gate": mat(ff, d),
                                "b_ff_gate": vec(ff, 0.0), "w_ff2": mat(d, ff), "b_ff2": vec(d, 0.0)})
        cfg = grilly_amd.PreNormEncoderConfig(layers=layers, d_model=d, heads=heads, d_ff=ff, vocab=vocab)
        return grilly_amd.PreNormEncoder(_backend(), cfg, w, dtype=case["dtype"])
    w.update(pos_emb=mat(512, d), type_emb=mat(2, d))
    for _ in range(layers):
        w["layers"].append({"w_qkv": mat(3 * d, d), "b_qkv": vec(3 * d, 0.0), "w_o": mat(d, d), "b_o": vec(d, 0.0), "ln1_g": vec(d, 1.0),
                            "ln1_b": vec(d, 0.0), "w_ff1": mat(ff, d), "b_ff1": vec(ff, 0.0), "w_ff2": mat(d, ff), "b_ff2": vec(d, 0.0),
                            "ln2_g": vec(d, 1.0), "ln2_b": vec(d, 0.0)})
    cfg = grilly_amd.EncoderConfig(layers=layers, d_model=d, heads=heads, d_ff=ff, vocab=vocab)
    return grilly_amd.BertEncoder(_backend(), cfg, w, dtype=case["dtype"])


def prepare(case, seed):
    family, dtype = case["family"], case["dtype"]
    state = {"case": case, "backend": _backend()}
    if family == "encoder":
        rng = np.random.default_rng(seed)
        state["encoder"] = _encoder(case, seed)
        state["ids"] = rng.integers(0, ARCHS[case["arch"]][4], (case["b"], case["s"])).astype(np.int64)
        # a tokenizer hands over a mask with every batch, all ones where nothing is padded
        n = _padded_lengths(rng, case) if case["pad"] else np.full(case["b"], case["s"])
        state["mask"] = (np.arange(case["s"])[None, :] < n[:, None]).astype(np.int64)
        return state
    normal = _normals(seed)
    if family == "fnn":
        m, k, n = case["m"], case["k"], case["n"]
        state["x"] = normal((m, k)).cpu().numpy()
        std = 1.0 / math.sqrt(k)
        state["w"] = normal((n, k), std).cpu().numpy()
        state["b"] = normal((n,), 0.02).cpu().numpy()
        if case["op"] == "fused_swiglu":
            state["w_up"] = normal((n, k), std).cpu().numpy()
            state["b_up"] = normal((n,), 0.02).cpu().numpy()
        return state
    storage = torch.bfloat16 if dtype == "bf16" else torch.float32
    if family == "mlp":
        m, k, n = case["m"], case["k"], case["n"]
        state["x"] = normal((m, k)).to(storage)
        state["w_gate"], state["w_up"] = normal((n, k), 0.02).to(storage), normal((n, k), 0.02).to(storage)
        state["w_down"] = normal((k, n), 0.02).to(storage)
        state["hidden"], state["y"] = torch.empty(m, n, dtype=storage, device="cuda"), torch.empty(m, k, dtype=storage, device="cuda")
        return state
    q, k, v = (normal((case["b"], case["s"], case["h"], case["d"])) for _ in range(3))
    if family == "attention":
        state.update(q=q.cpu().numpy(), k=k.cpu().numpy(), v=v.cpu().numpy())
    else:
        state.update(q=q.to(storage), k=k.to(storage), v=v.to(storage), o=torch.empty(q.shape, dtype=storage, device="cuda"))
    return state


# ---------------------------------------------------------------------------------------------- one pass
def run(state):
    case, backend = state["case"], state["backend"]
    family, dtype = case["family"], case["dtype"]
    if family == "encoder":
        return state["encoder"].forward(state["ids"], state["mask"], pool=case["pool"])
    if family == "fnn":
        if case["op"] == "fused_swiglu":
            return backend.fnn.fused_swiglu(state["x"], state["w"], state["w_up"], state["b"], state["b_up"], dtype=dtype)
        op = backend.fnn.linear if case["op"] == "linear" else backend.fnn.fused_linear_gelu
        return op(state["x"], state["w"], state["b"], dtype=dtype)
    if family == "attention":
        op = backend.attention.flash_attention2_rope if case["rope"] else backend.attention.flash_attention2
        return op(state["q"], state["k"], state["v"], case["h"], case["d"], causal=case["causal"], dtype=dtype)
    c, code = backend.core, dtype_code(dtype)
    if family == "mlp":
        m, k, n = case["m"], case["k"], case["n"]
        L.check(c.lib.grl_swiglu_nt(c.ctx, code, code, m, n, k, state["x"].data_ptr(), state["w_gate"].data_ptr(), state["w_up"].data_ptr(),
                                    None, None, state["hidden"].data_ptr(), None, None), "swiglu_nt")
        L.check(c.lib.grl_gemm_nt(c.ctx, code, code, m, k, n, state["hidden"].data_ptr(), state["w_down"].data_ptr(), None,
                                  state["y"].data_ptr(), L.EPI_NONE), "gemm_nt")
        return {"hidden": state["hidden"], "y": state["y"]}
    L.check(c.lib.grl_fa2_fwd(c.ctx, code, case["b"], case["s"], case["h"], case["d"], state["q"].data_ptr(), state["k"].data_ptr(),
                              state["v"].data_ptr(), None, state["o"].data_ptr(), 1.0 / math.sqrt(case["d"]), int(case["causal"]),
                              L.ROPE_INTERLEAVED if case["rope"] else L.ROPE_NONE, 10000.0, 1.0, None), "fa2_fwd")
    return state["o"]


# ---------------------------------------------------------------------------------------------- what a pass needs
def work(case):
    """Bytes: each input once, each output once (numpy arrays at their own four bytes a value, ids and mask at eight).
    FLOPs: two per multiply-add of the products, half of the scores where the causal rule drops them; of a padded batch
    only the real tokens count where only pooled embeddings come back (at the mean of the lengths' distribution)."""
    family, es = case["family"], _es(case)
    if family == "fnn":
        m, k, n = case["m"], case["k"], case["n"]
        mats = 2 if case["op"] == "fused_swiglu" else 1
        return {"bytes": 4.0 * (m * k + mats * n * (k + 1) + m * n), "flops": 2.0 * mats * m * k * n}
    if family == "mlp":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": float(es) * (2 * m * k + 3 * k * n + 2 * m * n), "flops": 6.0 * m * k * n}
    if family in ("attention", "device_attention"):
        elems = float(case["b"]) * case["s"] * case["h"] * case["d"]
        return {"bytes": 4.0 * elems * (4 if family == "attention" else es), "flops": 4.0 * elems * case["s"] * (0.5 if case["causal"] else 1.0)}
    layers, d, heads, ff, vocab = ARCHS[case["arch"]]
    b, s = case["b"], case["s"]
    mean, square = float(s), float(s) * s
    if case["pad"] and case["pool"]:
        lo = max(1, s // 8)
        mean, square = (lo + s) / 2.0, (s ** 3 - lo ** 3) / (3.0 * (s - lo)) if s > lo else float(s) * s
        mean, square = (mean * (b - 1) + s) / b, (square * (b - 1) + s * s) / b
    mlp = (3 if case["arch"] == "prenorm" else 2) * d * ff
    tokens = b * mean
    flops = layers * (2.0 * tokens * (4 * d * d + mlp) + 4.0 * b * square * d)
    out = 4.0 * b * d * (1 if case["pool"] else s)
    rows = min(tokens, vocab)
    return {"bytes": layers * float(es) * (4 * d * d + mlp) + 4.0 * rows * d + 16.0 * b * s + out, "flops": flops}


def tolerance(case):
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    # one bf16 rounding of operands and results; through a stack of layers the hidden states are rounded six times a layer
    return {"rel": 2e-2 if case["family"] == "encoder" else 1e-2}
