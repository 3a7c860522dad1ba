"""What the compiler makes of the transfers written in inline assembly, read from the assembly of a small kernel built here (no GPU)."""
import glob
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "grilly_amd", "csrc")
SOURCE = r"""
#include "common.hpp"
__global__ void transfers(const void* p, int* out, int n) {
    __shared__ __attribute__((aligned(1024))) char lds[4096];
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, n, 0x00020000);
    auto own = [&](int at) { __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)lds, 16, threadIdx.x * 16, at, 0, 0); };
    own(4096);
    dma16(make_rsrc_words(p, n), 1024, threadIdx.x * 16, n, 64);
    own(8192);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    out[threadIdx.x] = ((int*)lds)[threadIdx.x];
}
"""


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    at = tmp_path_factory.mktemp("asm")
    (at / "t.hip").write_text(SOURCE)
    subprocess.run(["hipcc", "-std=c++17", "-O3", "--offload-arch=gfx950", "--offload-device-only", "-S", "-Wno-unused-result", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-I", CSRC, "-o", str(at / "t.s"), str(at / "t.hip")], check=True, timeout=100)
    lines = [l.split(";")[0].strip() for l in (at / "t.s").read_text().splitlines()]
    return [l for l in lines if l and not l.startswith(".")]


def test_every_transfer_has_its_destination(code):
    """The compiler's own transfer behind the inline one sets m0 again, where both of its transfers go to the same place."""
    at = [i for i, l in enumerate(code) if re.match(r"buffer_load_dwordx4 .* lds$", l)]
    assert len(at) == 3
    for first, last in zip([-1] + at, at):
        assert any(re.match(r"s_\w+ m0,", l) for l in code[first + 1:last]), code


def test_a_wait_state_follows_the_write_of_m0(code):
    """as the compiler arranges it for its own transfers"""
    for i, l in enumerate(code):
        if re.match(r"s_\w+ m0,", l):
            assert not code[i + 1].endswith(" lds"), code[i:i + 2]


def test_one_place_writes_m0():
    text = "".join(open(f).read() for pattern in ("*.hip", "*.hpp") for f in glob.glob(os.path.join(CSRC, pattern)))
    assert len(re.findall(r"s_mov_b32 m0", text)) == 1
