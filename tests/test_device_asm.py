"""What the compiler makes of the transfers written in inline assembly, read from the assembly of a small kernel built here and from that of
the library as built (no GPU)."""
import glob
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

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


def scalars(operand):
    m = re.match(r"s\[(\d+):(\d+)\]$|s(\d+)$", operand)
    return frozenset() if not m else frozenset(range(int(m[1]), int(m[2]) + 1)) if m[1] else frozenset([int(m[3])])


def written(code, unit):
    """scalar registers that an instruction of the vector ("v_") or the scalar ("s_") unit writes"""
    name, _, rest = code.partition(" ")
    operands = [o.strip() for o in rest.split(",")]
    if not name.startswith(unit) or unit == "s_" and name.startswith(("s_cmp", "s_cbranch", "s_bitcmp", "s_branch", "s_waitcnt", "s_nop", "s_barrier")):
        return frozenset()
    return scalars(operands[0]) | (scalars(operands[1]) if unit == "v_" and len(operands) > 1 and re.match(r"v_\w+_co|v_div_scale|v_mad_[iu]64", name) else frozenset())


def short_waits(kernel):
    """(number of transfers to LDS, those whose scalars are not there yet).  A transfer needs one wait state behind a scalar write of m0, and five
    behind a write of its resource or offset by the vector unit; no interlock stands in, and the compiler counts for its own ones only."""
    jumps, bad = {}, []
    for i, l in enumerate(kernel):
        if l.startswith(("s_cbranch", "s_branch")):
            jumps.setdefault("<" + l.split()[-1] + ">:", []).append(i)
    at = [i for i, l in enumerate(kernel) if l.startswith("buffer_load") and l.endswith(" lds")]
    for i in at:
        if re.match(r"s_\w+ m0,", kernel[i - 1]):
            bad.append(kernel[i - 1:i + 1])
        reads = frozenset().union(*(scalars(o.strip().split(" ")[0]) for o in kernel[i].partition(" ")[2].split(",")[1:]))
        todo, seen = [(i - 1, 0, reads)], set()
        while todo:
            j, states, need = todo.pop()
            while j >= 0 and states < 5 and need and (j, states, need) not in seen:
                seen.add((j, states, need))
                l = kernel[j]
                if l.startswith("<"):
                    todo += [(k, states, need) for k in jumps.get(l, [])]
                    if kernel[j - 1].startswith(("s_branch", "s_endpgm")):
                        break
                elif written(l, "v_") & need:
                    bad.append([l, kernel[i], states])
                    break
                else:
                    need -= written(l, "s_")
                    states += int(l.split()[1]) + 1 if l.startswith("s_nop") else 1
                j -= 1
    return len(at), bad


def test_the_check_sees_a_short_wait():
    load = "buffer_load_dwordx4 v3, s[4:7], s9 offen lds"
    assert short_waits(["s_mov_b32 m0, s1", load])[1] and not short_waits(["s_mov_b32 m0, s1", "s_add_i32 s9, s2, s3", load])[1]
    assert short_waits(["v_readfirstlane_b32 s6, v1", "s_nop 1", "s_nop 1", load])[1] and not short_waits(["v_readfirstlane_b32 s6, v1", "s_nop 4", load])[1]
    assert not short_waits(["v_mad_u64_u32 v[0:1], s[8:9], v2, v3, 0", "s_add_i32 s9, s2, s3", load])[1]
    assert short_waits(["s_mov_b32 m0, s1", "<L1>:", "s_nop 0", load, "v_readlane_b32 s5, v9, 3", "s_cbranch_scc1 L1"])[1]


def test_every_transfer_of_the_library_has_its_waits(tmp_path):
    llvm, lib = "/opt/rocm/llvm/bin/llvm-objdump", os.path.join(os.path.dirname(CSRC), "lib", "libgrilly_hip.so")
    if not os.path.exists(lib):
        pytest.skip("library not built")
    shutil.copy(lib, tmp_path / "l.so")
    subprocess.run([llvm, "--offloading", "l.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL, timeout=60)

    def disassemble(path):
        text = subprocess.run([llvm, "-d", "--symbolize-operands", "--no-show-raw-insn", "--no-leading-addr", path], check=True, capture_output=True, text=True, timeout=100).stdout
        return [k for k in re.split(r"^<_\S+>:$", text, flags=re.M)[1:] if " lds " in k]
    transfers = 0
    with ThreadPoolExecutor(4) as pool:
        for kernels in pool.map(disassemble, sorted(glob.glob(str(tmp_path / "*gfx950")))):
            for k in kernels:
                n, bad = short_waits([l for l in (l.split("//")[0].strip() for l in k.splitlines()) if l])
                assert not bad, bad[:3]
                transfers += n
    assert transfers > 1000


def test_phased_kernels_keep_nothing_in_scratch(tmp_path):
    """A reload from scratch waits for the wave's memory counter to run out, the transfers of two steps with it."""
    llvm, lib = "/opt/rocm/llvm/bin", os.path.join(os.path.dirname(CSRC), "lib", "libgrilly_hip.so")
    if not os.path.exists(lib):
        pytest.skip("library not built")
    shutil.copy(lib, tmp_path / "l.so")
    subprocess.run([os.path.join(llvm, "llvm-objdump"), "--offloading", "l.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL, timeout=60)
    scratch = {}
    for f in glob.glob(str(tmp_path / "*gfx950")):
        notes = subprocess.run([os.path.join(llvm, "llvm-readelf"), "--notes", f], check=True, capture_output=True, text=True, timeout=60).stdout
        for k in re.split(r"\n  - ", notes):
            name, size = re.search(r"\.name:\s+(\S+)", k), re.search(r"\.private_segment_fixed_size:\s+(\d+)", k)
            if name and size and "gemm_nt_phased_kernel" in name[1]:
                scratch[name[1]] = int(size[1])
    assert len(scratch) > 10 and not any(scratch.values()), scratch
