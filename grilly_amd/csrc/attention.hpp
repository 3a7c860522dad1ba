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
// the XCDs in turn (in place of 1: mixed, some heads would be computed twice and others never), 8 (ragged batches, on top of 4) the longest
// sequences first.
static inline int fa_order_checked(int order) { return order & 4 ? order & 14 : order & 3; }
constexpr int FA_MOST_RANKED = 32;        // sequences of a batch that a workgroup ranks by length
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
// Dealt-out ragged batches of few long sequences of unequal length: the longest first.  Their workgroups (`blocks` of 128 queries, empty ones
// counted) are all resident at once or nearly, so a launch lasts as long as the CU that was dealt the most work; by falling length the deal
// comes out nearly even.  Every workgroup ranks the sequences for itself, which costs a launch 0.5 to 1.5 us.  In batch order / ranked, mean
// of 26 sizes (8 .. 32 sequences, longest 260 .. 1024, 8 .. 16 heads of 64 and 128), by how full the rectangle B x S is: 0.43 0.93, 0.58 0.94,
// 0.76 0.99, 0.86 1.003, 0.93 1.02, 1.0 1.03.  us, lengths uniform from an eighth to all of S: 32 x 300 x 12 heads of 64 18.2 -> 17.0, 24 x 300 x 12
// 16.7 -> 13.7, 16 x 512 x 12 18.4 -> 17.4, 13 x 749 x 12 28.4 -> 19.5, 24 x 900 x 8 39.3 -> 36.6, 32 x 400 x 8 heads of 128 35.0 -> 32.5.
// Where the line leaves off: rectangles more than three quarters full (32 x 300 x 12 all of 300: 24.3 -> 25.7), fewer blocks than 2.5 per CU are no
// deal (10 x 512 x 8 12.1 -> 13.1), short sequences lose the ranking's time (24 x 200 x 12 11.3 -> 11.5), so do causal ones up to 512, whose
// work falls off with the square of the length (30 x 465 x 12 heads of 128 36.5 -> 39.4), sequences of four blocks gain nothing once they are more
// than four blocks per CU (24 x 512 x 12 1.02, 21 x 476 x 16 1.03, 28 x 512 x 16 0.995; of three blocks 32 x 384 x 12 0.89, of six and more 0.93),
// and of many blocks or sequences the later ones fill the gaps as they come (64 x 512 x 12 49.9 -> 52.6, 32 x 900 x 16 73.2 -> 74.5).
static inline int fa_order_ranked(int order, bool causal, int64_t S, int64_t B, int64_t H, int64_t rows, int64_t cus) {
    const int64_t each = (S + 127) / 128, blocks = B * H * each;
    return order == 4 && S > (causal ? 512 : 256) && B > 1 && B <= FA_MOST_RANKED && 4 * rows <= 3 * B * S && 2 * blocks >= 5 * cus && blocks <= (each == 4 ? 4 : 12) * cus ? 12 : order;
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

typedef __attribute__((ext_vector_type(4))) int i32x4_t;

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

// Where a sequence of `len` rows stands among those of its batch, larger keys first: the longest first, of equal ones the first in the batch.
// Distinct and not negative whatever `len` is (offsets that fall count as empty sequences): every rank below B has its owner.
__host__ __device__ __forceinline__ int fa_rank_key(int len, int b) {
    return (len < 0 ? 0 : len < 65536 ? len : 65536) * FA_MOST_RANKED + FA_MOST_RANKED - 1 - b;
}
// The sequence of the given rank: b, its first row and its length.
// `scratch`: LDS of at least FA_MOST_RANKED + 4 ints that nobody else writes before the workgroup meets again behind this.
template <int NT> __device__ __forceinline__ void fa_ranked(const int32_t* offsets, int B, int rank, int* scratch, int& b, int64_t& row0, int& len) {
    const int tid = threadIdx.x, B4 = (B + 3) & ~3;
    int mine = 0, first = 0, own = 0;
    if (tid < B4) {
        if (tid < B) {
            first = offsets[tid];
            own = offsets[tid + 1] - first;
            mine = fa_rank_key(own, tid);
        }
        scratch[tid] = mine;             // 0 behind the batch
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (tid < B) {
        int longer = 0;
        for (int u = 0; u < B4; u += 4) {
            const i32x4_t v = *(const i32x4_t*)(scratch + u);
#pragma unroll
            for (int e = 0; e < 4; ++e) longer += v[e] > mine;
        }
        if (longer == rank) *(i32x4_t*)(scratch + FA_MOST_RANKED) = i32x4_t{tid, first, own, 0};
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const i32x4_t found = *(const i32x4_t*)(scratch + FA_MOST_RANKED);
    b = __builtin_amdgcn_readfirstlane(found[0]);
    row0 = __builtin_amdgcn_readfirstlane(found[1]);
    len = __builtin_amdgcn_readfirstlane(found[2]);
}

template <int N, typename F> __device__ __forceinline__ void sfor(F&& f) {
    if constexpr (N > 0) {
        sfor<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// fp32 operands, head dims 32 / 64 / 128 (attention_f32.hip); rope: interleaved pairs, rotated as the rows are loaded
int launch_fa32(grl_ctx* c, const FaArgs& a, int D, bool rope);
