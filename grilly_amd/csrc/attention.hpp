// What the two Flash-Attention-2 kernels (attention.hip: bf16, attention_f32.hip: fp32) share.
#pragma once
#include "common.hpp"
#include <type_traits>

struct FaArgs {
    const void* Q; const void* K; const void* V;
    const float* mask;        // (B,S) or null
    const int32_t* offsets;   // first row of each sequence of a ragged batch (B+1 entries; S is then the longest length), or null
    const int32_t* positions; // ragged batch: position of each row in its sequence
    void* O;
    const float2* rope;       // (S, D/2) {cos, sin} or null
    int B, S, H;
    float scale;
    int causal;
    int64_t q_stride, k_stride, v_stride, o_stride;   // elements between consecutive positions
};

// Workgroup numbering of the bf16 kernel, bits: 1 XCD-contiguous runs of ids, 2 the heaviest query blocks of all heads first, 4 heads dealt out to
// the XCDs in turn (in place of 1: mixed, some heads would be computed twice and others never).
static inline int fa_order_checked(int order) { return order & 4 ? order & 6 : order & 3; }
// Measured: causal and short sequences do best head by head on XCD-contiguous runs; long dense sequences with the plain id order (32 CUs of
// an XCD streaming the same K/V tiles in lockstep miss L2 together).
// Ragged batches (without mask and rotation: see the kernel): heads dealt out.  A contiguous run per XCD gives an XCD six sequences of a
// batch of 48, and the launch lasts as long as the longest six (48 sequences up to 384 long, 12 heads: 30.9 -> 28.5 us; 32 up to 300:
// 20.0 -> 19.7; 16 to 128 sequences of 16 to 900 tokens, 4 to 16 heads: 4 % on the mean at head dim 64, 3 % at 128).  Not at head dim 32: two heads
// share every 128-byte line of K and V, which then goes to two XCDs (64 sequences 2 % slower on the mean, 128 sequences 8 %, of equal
// length up to 46 %).  A rectangular batch with a mask is level to 5 % slower (32 x 200), and with few heads a turn is too coarse.
static inline int fa_order(bool causal, int64_t S, bool ragged, int64_t heads, int D) {
    if (ragged && D >= 64 && heads >= 64 && S <= 1024) return 4;
    return causal || S <= 1024 ? 1 : 0;
}
// Where workgroup `id` of nwg = nqb * nbh stands in the walk.  DEAL: the heads that make whole turns of eight are dealt out, the query blocks
// of one head next to each other on one XCD; the rest keep their ids.
template <bool DEAL> __host__ __device__ __forceinline__ int fa_place(int order, int id, int nwg, int nqb, int nbh) {
    const int per = nwg >> 3, rem = nwg & 7, xcd = id & 7, loc = id >> 3;
    int lin = (order & 1) ? xcd * per + (xcd < rem ? xcd : rem) + loc : id;
    if constexpr (DEAL)
        if ((order & 4) && id < (nbh & ~7) * nqb) lin = (loc / nqb * 8 + xcd) * nqb + loc % nqb;
    return lin;
}

// Sequence b of the batch: its first row and its length.  In a ragged batch the sequences stand back to back and every one
// has its own length (queries and keys alike); the grid is laid out for the longest, and a workgroup whose queries lie past
// the end of its sequence has nothing to do.
__device__ __forceinline__ void fa_sequence(const int32_t* offsets, int b, int S, int64_t& row0, int& len) {
    if (offsets) {
        const int o = __builtin_amdgcn_readfirstlane(offsets[b]), e = __builtin_amdgcn_readfirstlane(offsets[b + 1]);
        row0 = o; len = e - o;
    } else {
        row0 = (int64_t)b * S; len = S;
    }
}

template <int N, typename F> __device__ __forceinline__ void sfor(F&& f) {
    if constexpr (N > 0) {
        sfor<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// fp32 operands, head dims 32 / 64 / 128 (attention_f32.hip); rope: interleaved pairs, rotated as the rows are loaded
int launch_fa32(grl_ctx* c, const FaArgs& a, int D, bool rope);
