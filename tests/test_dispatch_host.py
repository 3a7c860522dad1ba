"""The launchers' host rules, compiled from the kernels' headers by the host pass alone (no GPU, no device code)."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "grilly_amd", "csrc")
SOURCE = r"""
#include "gemm_kernels.hpp"
#include "attention.hpp"
extern "C" int kernel_run(int variant, int elem_size, int dual) { return gemm_kernel_run(variant, elem_size, dual); }
extern "C" int kernel(long long M, long long N, long long K, int elem_size, int dual) { return gemm_kernel(M, N, K, elem_size, dual, 256); }
extern "C" int product(long long M, long long N, long long K, int shares) { return gemm_kernel(M, N, K, 4, false, 256, 0, (Shares)shares); }
extern "C" int rope_kernel(long long M, long long N, long long K, int elem_size) { return gemm_rope_kernel(M, N, K, 2 * N / 3, elem_size, 256); }
extern "C" int resln_kernel(long long M, long long N, long long K, int elem_size) { return gemm_resln_kernel(M, N, K, elem_size, 256); }
extern "C" int takes_partials(int kernel) { return gemm_kernel_takes_partials(kernel); }
extern "C" int order_checked(int order) { return fa_order_checked(order); }
extern "C" int order(int causal, int S, int ragged, int heads, int D) { return fa_order(causal, S, ragged, heads, D); }
extern "C" int ranked(int order, int causal, int S, int B, int H, long long rows, int cus) { return fa_order_ranked(order, causal, S, B, H, rows, cus); }
extern "C" int rank_key(int len, int b) { return fa_rank_key(len, b); }
extern "C" int place(int deal, int order, int id, int nwg, int nqb, int nbh) {
    return deal ? fa_place<true>(order, id, nwg, nqb, nbh) : fa_place<false>(order, id, nwg, nqb, nbh);
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    at = tmp_path_factory.mktemp("rules")
    (at / "rules.hip").write_text(SOURCE)
    subprocess.run(["hipcc", "-std=c++17", "-O0", "--offload-host-only", "-shared", "-fPIC", "-Wno-unused-result", "-I", CSRC,
                    "-o", str(at / "rules.so"), str(at / "rules.hip")], check=True, timeout=100)
    lib = ctypes.CDLL(str(at / "rules.so"))
    lib.kernel.argtypes = [ctypes.c_longlong] * 3 + [ctypes.c_int] * 2
    lib.ranked.argtypes = [ctypes.c_int] * 5 + [ctypes.c_longlong, ctypes.c_int]
    lib.product.argtypes = [ctypes.c_longlong] * 3 + [ctypes.c_int]
    lib.rope_kernel.argtypes = lib.resln_kernel.argtypes = [ctypes.c_longlong] * 3 + [ctypes.c_int]
    return lib


@pytest.mark.parametrize("elem_size", [2, 4])
@pytest.mark.parametrize("dual", [0, 1])
def test_partials_go_to_kernels_that_merge_them(rules, elem_size, dual):
    """The shared-K kernels (9, 10) and the register-staged ones (1, 2, 5) read merged statistics from memory: no number may end in one of
    them and count as a kernel that takes partials."""
    has = {1, 2, 3, 4, 5, 9} | ({6, 7, 8} if elem_size == 2 and not dual else {6, 7} if elem_size == 4 else set())
    has |= {10} if elem_size == 2 else {11}
    has |= {8} if elem_size == 4 and not dual else set()
    for variant in range(1, 12):
        kernel = rules.kernel_run(variant, elem_size, dual)
        assert kernel in has and (variant not in has or kernel == variant)
        assert rules.takes_partials(kernel) == (kernel in (3, 4, 6, 7, 8))


@pytest.mark.parametrize("order", range(8))
def test_every_attention_block_is_computed_once(rules, order):
    """whatever GRL_FA_ORDER says, in the kernels with and without the dealt-out map"""
    order = rules.order_checked(order)
    for deal in (0, 1):
        for nbh in (1, 7, 8, 9, 24, 70):
            for nqb in (1, 2, 3, 8):
                n = nbh * nqb
                assert sorted(rules.place(deal, order, i, n, nqb, nbh) for i in range(n)) == list(range(n))


def test_heads_that_share_lines_are_not_dealt_out(rules):
    """head dim 32: two heads in every 128-byte line, which dealing out would send to two XCDs"""
    assert [rules.order(0, 256, 1, 1536, D) for D in (32, 64, 128)] == [1, 4, 4]
    assert rules.order(0, 1025, 1, 1536, 64) == 0 and rules.order(1, 4096, 0, 64, 128) == 1


def test_two_shared_tiles_per_unit_need_a_long_sum(rules):
    """bf16: between 257 and 512 tiles of 64 x 64 the shared-K kernel is ahead everywhere from 96 slabs on only"""
    for M, N in ((2100, 512), (2600, 512), (1088, 1152), (2000, 768), (512, 4096)):
        assert [rules.kernel(M, N, K, 2, 0) for K in (3072, 5120, 6080, 6144, 11008)] == [8, 8, 8, 10, 10]
    assert rules.kernel(800, 768, 768, 2, 0) == 10


def test_rotary_products(rules):
    """which kernel rotates in its epilogue; 0: none, and no table is fetched for it"""
    assert [rules.rope_kernel(M, 2304, 768, 2) for M in (16, 100, 400, 810, 1500, 3000, 5390, 65536)] == [9, 9, 10, 7, 6, 4, 3, 3]
    assert [rules.rope_kernel(M, 2304, 768, 4) for M in (27, 300, 3000, 65536)] == [9, 9, 0, 0]
    assert rules.rope_kernel(100, 2304, 776, 2) == 0 and rules.rope_kernel(100, 96, 768, 2) == 0


def test_sizes_of_the_row_partials_tests(rules):
    """test_gpu_row_partials names the bf16 kernel that writes the partials and the one that merges them; both as the launchers choose."""
    from test_gpu_row_partials import GATED, LAYERS
    for M, d, ff, writes, reads in GATED:
        assert rules.resln_kernel(M, d, d, 2) == writes and rules.kernel(M, ff, d, 2, 1) == reads, (M, d)
    for B, S, heads, ff, kernels in LAYERS:
        M, d = B * S, 64 * heads
        assert (rules.resln_kernel(M, d, d, 2), rules.resln_kernel(M, d, ff, 2), rules.kernel(M, 3 * d, d, 2, 0), rules.kernel(M, ff, d, 2, 0)) == kernels, (M, d)
    assert {g[3] for g in GATED} == {3, 4, 6, 7} and {k for l in LAYERS for k in l[4]} >= {3, 4, 6, 7, 8}
    odd = [(M, d, w) for M, d, _, w, _ in GATED if M % 2 and 128 < d <= (1536 if w == 3 else 768)]      # two to six partials
    assert {w for _, _, w in odd} == {3, 4, 6, 7}


NEVER, NOT_NOW, YES = 0, 1, 2          # enum class Shares


def test_recorded_products_are_no_less_accurate(rules):
    """fp32 under capture: what is far better off in shares of K takes kernel 6, whose four chains the shares are, not the fastest kernel
    without shares (3 or 4: one chain; 9 on the fp32 instruction).  Kernel 9 stays where it is no more than somewhat behind the shares."""
    far = [(4128, 2304, 8192), (4419, 2048, 6144), (2091, 8192, 8192), (5971, 1152, 6144), (230, 1536, 10400), (8, 1536, 7136), (1500, 768, 3072)]
    assert [rules.product(*s, YES) for s in far] == [11] * 7 and [rules.product(*s, NOT_NOW) for s in far] == [6] * 7
    assert {3, 4, 9} == {rules.product(*s, NEVER) for s in far[:-1]}
    near = [(450, 768, 3072), (350, 768, 3072), (1200, 512, 2048)]
    assert [rules.product(*s, YES) for s in near] == [11] * 3 and [rules.product(*s, NOT_NOW) for s in near] == [9] * 3
    for M in range(8, 6000, 83):
        for N in (128, 384, 768, 1152, 2304, 4096):
            for K in (480, 512, 1152, 3072, 8192):
                assert rules.product(M, N, K, NOT_NOW) in (6, rules.product(M, N, K, NEVER))


def test_shares_of_k_in_place_of_two_small_tiles_a_unit(rules):
    """(M, N, K): 11 only where a unit gets two 32 x 32 tiles or more of 1024 k at least, each line from both sides"""
    sizes = [(300, 768, 3072), (351, 768, 3072), (639, 768, 3072), (449, 1024, 4096), (1201, 512, 2048),
             (1999, 764, 1152), (1753, 764, 1152), (1688, 764, 1024), (1688, 764, 992), (566, 1800, 896), (563, 2048, 896), (349, 3072, 960)]
    assert [rules.product(*s, YES) for s in sizes] == [9, 11, 11, 11, 11, 9, 11, 11, 9, 9, 9, 9]
    assert {rules.product(*s, NEVER) for s in sizes} == {9} and rules.product(33, 388, 2080, YES) == 9


@pytest.mark.parametrize("lens", [[5, 0, 900, 5, 900, 1, 0], [-7, 3, -2 ** 31, 0, 3, -1], [2 ** 31 - 1, 65536, 65537, 1, 2 ** 26], [300] * 32, [-1] * 31 + [0], list(range(32, 0, -1))])
def test_every_rank_has_one_sequence(rules, lens):
    """as fa_ranked counts: the longer ones among the batch and the zeros that fill its last four.  Lengths as any offsets give them, also falling ones."""
    keys = [rules.rank_key(n, b) for b, n in enumerate(lens)]
    padded = keys + [0] * (-len(keys) % 4)
    ranks = [sum(k > mine for k in padded) for mine in keys]
    assert sorted(ranks) == list(range(len(lens)))
    length = lambda b: min(max(lens[b], 0), 65536)
    assert sorted(range(len(lens)), key=lambda b: ranks[b]) == sorted(range(len(lens)), key=lambda b: (-length(b), b))


@pytest.mark.parametrize("order", range(8, 16))
def test_every_block_is_computed_once_by_ranked_orders(rules, order):
    """GRL_FA_ORDER with the ranking's bit, which stands for nothing without dealt-out heads"""
    checked = rules.order_checked(order)
    assert checked & 8 == (8 if order & 4 else 0)
    test_every_attention_block_is_computed_once(rules, order)


def test_which_batches_are_ranked(rules):
    """both sides of each line: longest sequence, sequences, how full the rectangle is, blocks per compute unit, the order it stands on"""
    ranked = lambda S, B, H, fill=0.5, causal=0, order=4, cus=256: rules.ranked(order, causal, S, B, H, int(fill * B * S), cus) == 12
    assert ranked(300, 32, 12) and [ranked(S, 32, 12) for S in (256, 257)] == [False, True]
    assert [ranked(S, 16, 16, causal=1) for S in (512, 513)] == [False, True]
    assert [ranked(300, B, 16) for B in (32, 33)] == [True, False] and not ranked(1000, 1, 512)
    assert [ranked(600, 32, 12, fill) for fill in (0.75, 0.7501, 1.0)] == [True, False, False]
    assert [ranked(S, 32, H) for S, H in ((512, 8), (512, 9), (384, 9), (385, 9), (513, 9))] == [True, False, True, False, True]      # 1024 blocks, 1152, 864, 1152, 1440
    assert [ranked(384, B, H) for B, H in ((15, 14), (16, 14), (32, 8))] == [False, True, True]              # 630, 672, 768 blocks
    assert [ranked(512, 20, 8, cus=cus) for cus in (256, 257)] == [True, False] and [ranked(1024, 32, 12, cus=cus) for cus in (256, 255)] == [True, False]
    assert not any(ranked(300, 32, 12, order=order) for order in (0, 1, 2))


def test_one_phased_tile_for_each_unit(rules):
    """the size of the test of that name in test_gpu_gemm_phased: 256 x 256 tiles, fewer than compute units"""
    M, N = 71 * 256 - 37, 3 * 256 - 8
    assert all(rules.kernel(M, N, 64 * slabs, 2, 0) == 3 == rules.resln_kernel(M, N, 64 * slabs, 2) for slabs in (2, 3, 7))
