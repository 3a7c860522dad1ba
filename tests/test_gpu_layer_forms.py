"""Which layer form a BertEncoder batch runs by default: the lines themselves (CPU), and on the GPU that a batch between the five-launch
and the fused range is the seven-launch one bit for bit (in bf16 its hidden states are nearer to float64 than the fused form's)."""
import numpy as np
import pytest

from grilly_amd import BertEncoder, EncoderConfig, random_bert_weights
from grilly_amd import _lib as L


def test_fused_lines():
    for d in (64, 128, 384, 768, 1024, 4096):
        assert BertEncoder.fused_min_rows(d, L.GRL_BF16) == 8192
        rows = BertEncoder.fused_min_rows(d, L.GRL_F32)
        assert rows <= 8192 and (rows == 8192 or (rows - 1) * d < 3 << 20 <= rows * d)


def test_five_launch_line_looks_at_the_widest_product():
    for d, ff, rows in ((768, 3072, 768), (384, 1536, 1536), (768, 768, 1706), (256, 256, 5120), (768, 1536, 1024), (1024, 1024, 1280)):
        assert BertEncoder.rows_max(d, ff) == rows
        assert rows * max(3 * d, ff) <= 9 << 18 or rows * ff <= 5 << 18


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,B,S,heads", [("bf16", 30, 100, 12), ("bf16", 63, 130, 6), ("fp32", 30, 100, 12), ("fp32", 64, 127, 2)])
def test_batches_below_the_fused_line(backend, dtype, B, S, heads):
    cfg = EncoderConfig(layers=2, d_model=64 * heads, heads=heads, d_ff=256 * heads, vocab=100, max_pos=130)
    w = random_bert_weights(cfg, seed=3)
    ids = np.random.default_rng(1).integers(0, 100, (B, S))
    default, plain = BertEncoder(backend, cfg, w, dtype=dtype), BertEncoder(backend, cfg, w, dtype=dtype, fused=False)
    np.testing.assert_array_equal(default.forward(ids, pool=False), plain.forward(ids, pool=False))
