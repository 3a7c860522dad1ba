"""A process that gets no pinned host memory computes all the same, on the runtime's copies of pageable memory.  The refusal is
made on the host: a child process has a hipHostMalloc in front of the runtime's that hands out so many blocks and no more."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

REFUSE = """
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stdlib.h>
int refused;
int hipHostMalloc(void** p, size_t n, unsigned flags) {
    static int (*real)(void**, size_t, unsigned);
    static int handed;
    if (handed < atoi(getenv("PINNED_BLOCKS"))) {
        if (!real) real = (int (*)(void**, size_t, unsigned))dlsym(dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD), "hipHostMalloc");
        ++handed;
        return real(p, n, flags);
    }
    *p = 0;
    ++refused;
    return 2;      /* hipErrorOutOfMemory */
}
"""

CHILD = """
import ctypes, sys
refuse = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import numpy as np
import grilly_amd
from grilly_amd import BertEncoder, EncoderConfig, random_bert_weights
from grilly_amd import _lib as L
from oracle import oracle_np as O
backend = grilly_amd.Compute(0)
c = backend.core
rng = np.random.default_rng(0)
f = lambda *s: rng.standard_normal(s, dtype=np.float32)
for dtype, tol in (("fp32", 1e-4), ("bf16", 2e-2)):
    for m in (3, 700, 9000):                           # in place, slab, blocks
        x, w, b = f(m, 256), f(320, 256) / 16, f(320)
        for _ in range(2):
            assert O.max_rel(backend.fnn.linear(x, w, b, dtype=dtype), x @ w.T + b) < tol, (dtype, m)
    q, k, v = f(40, 64, 4, 64), f(40, 64, 4, 64), f(40, 64, 4, 64)
    got = backend.attention.flash_attention2(q, k, v, 4, 64, dtype=dtype)
    if dtype == "bf16":
        q, k, v = (O.bf16_round(t) for t in (q, k, v))
    assert O.max_rel(got[39:], O.truth_attention(q[39:], k[39:], v[39:])) < tol
    code = L.GRL_BF16 if dtype == "bf16" else L.GRL_F32
    for n in (5, 300000, 3000001):
        x = O.bf16_round(f(n)) if dtype == "bf16" else f(n)
        buf = c.upload(x, code)
        np.testing.assert_array_equal(c.download(buf, (n,), code), x)
        buf.free()
cfg = EncoderConfig(layers=1, d_model=64, heads=1, d_ff=128, vocab=50, max_pos=16)
enc = BertEncoder(backend, cfg, random_bert_weights(cfg), dtype="fp32")
ids = rng.integers(0, 50, (3, 16))
mask = (np.arange(16) < np.array([16, 4, 9])[:, None]).astype(np.int64)
assert np.isfinite(enc.forward(ids, mask)).all()
print("refused", ctypes.c_int.in_dll(refuse, "refused").value)
"""


@pytest.mark.gpu
@pytest.mark.parametrize("blocks", [0, 1, 2])
def test_without_pinned_memory(tmp_path, blocks):
    source, lib = tmp_path / "refuse.c", tmp_path / "refuse.so"
    source.write_text(REFUSE)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(source), "-ldl"], check=True)
    child = subprocess.run([sys.executable, "-c", CHILD, str(lib), ROOT], capture_output=True, text=True, timeout=100,
                           env=dict(os.environ, PINNED_BLOCKS=str(blocks)))
    assert child.returncode == 0, child.stdout + child.stderr
    assert "refused 1" in child.stdout          # asked once, then remembered
