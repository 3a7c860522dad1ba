// bf16 products on 256 x 256 tiles (with two weights: 256 x 128 outputs): persistent workgroups of eight waves, one per CU, whose K steps
// run in phases (included by gemm_kernels.hpp).
//
// A step is 64 k.  Its operands lie in one of two LDS stages of four halves, 128 rows each: A0, A1, B0, B1; half q holds the q-th 64
// activation rows of both wave rows, or the q-th 32 weight rows of the four wave columns (two weights: half 0 is the gate's, half 1 the
// up weight's).  A wave owns 128 x 64 of the tile and does a step in two phases: a memory part (fragment reads, transfers, a counted wait)
// and a matrix part of 32 instructions, a barrier behind each.  Waves 4 to 7 run one part behind waves 0 to 3, so that of the two waves of a
// SIMD one multiplies while the other reads.
//
//   memory part 0: reads B0, A0, B1 of step t;  requests A1 of step t + 1;          matrix part 0: rows of A0
//   memory part 1: reads A1 of step t;          requests B0, A0, B1 of step t + 2;  matrix part 1: rows of A1
//
// (X and Y below: Y is the operand whose halves are multiplied in turn, A, and X the other; with EPI_RESLN they change places.)
//
// A memory part ends when its reads are back, so a half is requested again one part after the waves behind have read it; the counted wait
// asks for it four parts later, and it is read six parts later.  64 to 96 KiB are in flight all the time.  The cursor runs on into the next tile,
// and the epilogue stands between the last matrix part and the next tile's first memory part; only A1 of the last step's stage is not
// being refilled then.  There, in the 2 KiB that its own transfers will fill, every wave turns 16 output rows at a time into 16-byte pieces of
// 128-byte rows: no barrier in the epilogue, and the stores stand behind the transfers of two steps in the memory counter.  An epilogue
// that only stores waits for none of them.  One that loads (residual, cos and sin) waits once for all that is in flight, because the
// counter retires in order.
//
// Bound: the board's power limit on real operands (with all-zero ones the same launches are 20 to 25 % faster: a step of 2048 matrix cycles
// takes 2340 at 2.4 GHz), then the output stores, which all CUs issue at once: without them 65536 x 2304 x 768 takes 163 us instead of
// 184, 65536 x 768 x 768 with LayerNormed residual 75 instead of 88.
// us, four phases of 16 instructions with an epilogue staged by the whole workgroup (four barriers, the stages drained for it) and the same LDS
// swizzle -> this, in turn on one box: 65536 x 2304 x 768 191.5 -> 183.7, folded 200.1 -> 190.3, 65536 x 1152 x 384 64.2 -> 61.2, folded 65536 x 3072 x
// 768 with GELU 297.4 -> 285.2, 65536 x 768 x 768 with LayerNormed residual 92.1 -> 91.3, 8192 x 8192 x 8192 747 -> 725, gated 16384 x 11008 x 4096
// 2050 -> 2023; 65536 x 768 x 3072 level.  Slower: bf16 residuals of short sums in several tiles (65536 x 768 x 128 44.0 -> 45.5, 33000 x 768 x 384
// 37.1 -> 37.7), whose epilogue that wait is most of.
// Without the stagger 27 % slower (four phases).  Tried and dropped: workgroups that start up to 3 us apart, so that their stores
// do not meet (65536 x 2304 x 768 184 -> 185; x 384 109 -> 106), stores that stay in the caches (188.7 -> 199.8), no wave priorities (level).
#pragma once

// ASKS: for launches of no more tiles than workgroups, see ask_for_residual
template <typename OutT, int EPI, bool DUAL, bool LN = false, bool ASKS = false>
__global__ __launch_bounds__(512) void gemm_nt_phased_kernel(GemmArgs p) {
    // A wave's share of the tile: 128 rows x 64 columns.  The row sums of EPI_RESLN are added chunk by chunk in the order of the 32 lanes that hold
    // a row of 256 columns elsewhere (c with c + 8, + 4, + 2, + 1, the halves last), which needs 128 columns of a row in one wave: 64 rows x
    // 128 columns there, weights and activations in each other's part.
    constexpr bool TR = EPI == EPI_RESLN;
    constexpr int BM = 256, BN = 256, BNO = DUAL ? BN / 2 : BN, WM = TR ? 64 : 128, WNO = TR ? 128 : BNO / 4, TNO = WNO / 32;
    constexpr int HALFB = 128 * 128, STAGE = 4 * HALFB;
    constexpr int OES = (int)sizeof(OutT), EPCO = 16 / OES;
    constexpr bool RL = EPI == EPI_RESLN;                   // LayerNorm(residual) formed in the epilogue + row statistics out
    constexpr bool HASRES = EPI == EPI_RES || RL, ROWS = LN || RL;
    // one tile's vectors, fp32: bias slice(s); with row statistics also the column sums c (c2), or the residual norm's beta, and the
    // tile's 256 row-statistics pairs.  Two buffers, alternating per tile.
    constexpr int VECS = 2 * STAGE, COLB = BN * 4, BIASB = ROWS ? 2 * COLB + BM * 8 : COLB;
    constexpr int PARTS_AT = VECS + 2 * BIASB, SUMS_AT = PARTS_AT + (ROWS ? GRL_MAX_PARTS * BM * 8 : 0);
    constexpr int ASKED_AT = SUMS_AT + (RL ? 2 * BM * 8 : 0);
    __shared__ __attribute__((aligned(1024))) char lds[ASKED_AT + (ASKS ? 1024 : 0)];
    static_assert(!ASKS || (HASRES && OES == 2), "what is asked for");
    static_assert(!(LN && RL) && !(RL && DUAL) && !(HASRES && DUAL), "one set of row statistics per tile");

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = TR ? wave >> 1 : wave >> 2, wn = TR ? wave & 1 : wave & 3, l4 = lane & 15, lq = lane >> 4;
    const bool behind = wave >= 4;                           // the waves that run one part behind
    const int ntiles = p.tiles_m * p.tiles_n;
    const int64_t rowbytes = (int64_t)p.K * 2;
    const int KT = p.K / 64;                                 // the host launches this kernel with two steps or more
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)lds;

    auto tile_of = [&](int pid, int& m0, int& n0) {          // as in gemm_nt_dma_kernel
        const int per = ntiles >> 3, rem = ntiles & 7, xcd = pid & 7, loc = pid >> 3;
        const int npid = xcd * per + (xcd < rem ? xcd : rem) + loc;
        const int width = p.group * p.tiles_n;
        const int first_m = (npid / width) * p.group;
        const int gsize = p.tiles_m - first_m < p.group ? p.tiles_m - first_m : p.group;
        m0 = (first_m + (npid % width) % gsize) * BM;
        n0 = ((npid % width) / gsize) * BNO;
    };
    auto rsrc_of = [&](const void* base, int first_row, int rows_total) {
        int64_t left = (int64_t)(rows_total - first_row) * rowbytes;
        if (left < 0) left = 0;
        return make_rsrc_words((const char*)base + (int64_t)first_row * rowbytes, left > 0xffffffffLL ? 0xffffffffu : (uint32_t)left);
    };

    // lane -> (row lr of an 8-row group, slot ls): LDS slot ls of row r holds chunk ls ^ lds_swz<8>(r)
    const int lr = lane >> 3, ls = lane & 7;
    const int lane_off[2] = {lr * (int)rowbytes + ((ls ^ lds_swz<8>(lr)) << 4), lr * (int)rowbytes + ((ls ^ lds_swz<8>(8 + lr)) << 4)};
    rsrc_words curA, curW, curW2, nextA, nextW, nextW2;
    int cur_k = 0, gstep = 0;                                // the cursor: byte of the row that is fetched next; steps done by this workgroup
    // this wave's two transfers of one half of the cursor's step into stage st: 16 rows, 2 KiB that no other wave fills
    auto issue_half = [&](auto ihalf, int st) {
        constexpr int h = decltype(ihalf)::value;
        constexpr bool isA = (h < 2) != TR;
        constexpr int q = h & 1;
        const int row = h < 2 ? (wave >> 2) * 128 + q * 64 + (wave & 3) * 16 : DUAL ? wave * 16 : (wave >> 1) * 64 + q * 32 + (wave & 1) * 16;
        const rsrc_words rs = isA ? curA : DUAL && q ? curW2 : curW;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int dst = (int)lds0 + (st & 1) * STAGE + h * HALFB + (wave * 16 + j * 8) * 128;
            dma16(rs, __builtin_amdgcn_readfirstlane(dst), lane_off[j], cur_k, (row + j * 8) * (int)rowbytes);
        }
    };
    using H_Y0 = std::integral_constant<int, 0>; using H_Y1 = std::integral_constant<int, 1>; using H_X0 = std::integral_constant<int, 2>; using H_X1 = std::integral_constant<int, 3>;
    auto advance = [&]() {
        cur_k += 128;
        if (cur_k == (int)rowbytes) { cur_k = 0; curA = nextA; curW = nextW; if constexpr (DUAL) curW2 = nextW2; }
    };
    // a tile's vectors: up to 1 KiB of `src` from a wave (columns and rows past the end read zero)
    auto fetch_vec = [&](const float* src, int left, int at, int bytes) {
        const int lane = EPI == EPI_ROPE ? fresh_lane() : (int)threadIdx.x & 63;
        rsrc_words rs = make_rsrc_words(src, left > 0 ? (uint32_t)left : 0u);
        asm volatile("s_nop 4" : "+s"(rs));             // the wait states behind a vector write of the words, where the compiler kept them in vector registers
        if (bytes >= 1024 || lane < bytes / 16) dma16(rs, __builtin_amdgcn_readfirstlane((int)lds0 + at), lane * 16, 0, 0);
    };
    auto issue_vectors = [&](int m0t, int n0t, int buf) {
        const int at = VECS + buf * BIASB, cols = (p.N - n0t) * 4, rows = (p.M - m0t) * 8;
        if (wave == 0 && p.bias) fetch_vec(p.bias + n0t, cols, at, BNO * 4);
        if (DUAL && wave == 4 && p.bias2) fetch_vec(p.bias2 + n0t, cols, at + BNO * 4, BNO * 4);
        if constexpr (ROWS) {
            if (wave == 1) fetch_vec((RL ? p.res_beta : p.ln_c) + n0t, cols, at + COLB, BNO * 4);
            if (DUAL && wave == 5) fetch_vec(p.ln_c2 + n0t, cols, at + COLB + BNO * 4, BNO * 4);
            if (p.nparts) {
                if (wave < p.nparts) {
                    const float* src = p.parts + 2 * ((int64_t)wave * p.M + m0t);
                    fetch_vec(src, rows, PARTS_AT + wave * BM * 8, 1024);
                    fetch_vec(src + 256, rows - 1024, PARTS_AT + wave * BM * 8 + 1024, 1024);
                }
            } else if (wave == 7) {
                const float* src = (RL ? p.res_stats : p.ln_stats) + 2 * (int64_t)m0t;
                fetch_vec(src, rows, at + 2 * COLB, 1024);
                fetch_vec(src + 256, rows - 1024, at + 2 * COLB + 1024, 1024);
            }
        }
    };
    static_assert(GRL_MAX_PARTS <= 8, "a wave per partial");

    OutT* C = (OutT*)p.C;
    const int rowB = p.N * OES;                             // bytes of an output row
    const bool staged = ((int64_t)p.N * OES) % 16 == 0 && !p.cache1 && !p.cache2 && (RL || (int64_t)p.N * OES * BM < (1LL << 31));
    constexpr int UB = WNO * OES >= 128 ? 128 : WNO * OES;  // bytes of a staged row
    constexpr int UC = UB / OES, GROUPS = WNO / UC, CB = UB / 16, PER = 16 * CB / 64;
    constexpr int UNITS = WM / 16 * GROUPS, STORES = UNITS * PER; // of a wave per tile
    static_assert(STORES + 8 < 64, "the memory counter's range");

    int pid = blockIdx.x, m0, n0, bbuf = 0;
    tile_of(pid, m0, n0);
    // A workgroup with one tile would do nothing but wait while its residual comes: the tile's lines are brought to L2 two steps before the end,
    // by transfers of 16 bytes of each (32 rows of four lines from a wave) into 1 KiB that nobody reads.  us, without -> with, no operand of
    // a launch touched by the one before: 16384 x 1024 x 1024 39.8 -> 36.5, with LayerNormed residual 44.3 -> 40.7, 18000 x 768 x 384 22.2 -> 21.1 and
    // 26.6 -> 25.6, 21000 x 768 x 768 32.1 -> 30.5 and 36.8 -> 34.7 (an epilogue staged by the whole workgroup: 37.1, 40.5, 20.8, 25.6, 31.1, 35.1).
    // A kernel of its own: with several tiles the lines push operands out of L2 (65536 x 2304 x 768 226 -> 241), and the test for it alone
    // spills scalars (1 % of 65536 x 768 x 768 with LayerNormed residual).  Six steps ahead is too early to find the lines there.
    auto ask_for_residual = [&] {
        const int64_t left = ((int64_t)(p.M - m0) * p.N - n0) * OES;
        rsrc_words rs = make_rsrc_words((const char*)p.residual + ((int64_t)m0 * p.N + n0) * OES, left > 0x7fffffff ? 0x7fffffffu : (uint32_t)left);
        asm volatile("s_nop 4" : "+s"(rs));                  // as in fetch_vec
        const int at = (wave * 32 + (lane >> 2)) * rowB + (lane & 3) * 128;
#pragma unroll
        for (int j = 0; j < 2; ++j) dma16(rs, __builtin_amdgcn_readfirstlane((int)lds0 + ASKED_AT), at, 0, 16 * j * rowB);
    };
    issue_vectors(m0, n0, bbuf);
    curA = rsrc_of(p.A, m0, p.M); curW = rsrc_of(p.W, n0, p.N);
    curW2 = DUAL ? rsrc_of(p.W2, n0, p.N) : curW;
    issue_half(H_X0{}, 0); issue_half(H_Y0{}, 0); issue_half(H_X1{}, 0); issue_half(H_Y1{}, 0);
    cur_k = 128;
    issue_half(H_X0{}, 1); issue_half(H_Y0{}, 1); issue_half(H_X1{}, 1);
    wait_vmcnt<6>();
    asm volatile("s_barrier" ::: "memory");
    if (behind) asm volatile("s_barrier" ::: "memory");
    bool stores_behind = false;                              // the previous tile's stores are behind the transfers that are due next
    int m0p = 0, n0p = 0;                                    // RL: the previous tile, whose row sums are still to be added
    bool sums_due = false;

    // RL: {sum, sum of squares} of a tile's rows from those of the two wave columns
    auto finish_rows = [&](int m0t, int n0t) {
        if constexpr (RL) {
            if (wave < 4) {
                const f32x2_t t = *(const f32x2_t*)(lds + SUMS_AT + tid * 8), u = *(const f32x2_t*)(lds + SUMS_AT + (BM + tid) * 8);
                if (m0t + tid < p.M) *(f32x2_t*)(p.part_out + ((int64_t)(n0t / BNO) * p.M + m0t + tid) * 2) = f32x2_t{t[0] + u[0], t[1] + u[1]};
            }
        }
    };
    // partials of the row statistics, merged in the first step: the same sums in the same order as ln_stats_merge_kernel
    auto merge_parts = [&] {
        if constexpr (ROWS) {
            if (p.nparts && wave < 4) {
                f32x2_t t[GRL_MAX_PARTS];
#pragma unroll
                for (int j = 0; j < GRL_MAX_PARTS; ++j) t[j] = *(const f32x2_t*)(lds + PARTS_AT + (j * BM + tid) * 8);
                float sum = 0.f, sq = 0.f;
#pragma unroll
                for (int j = 0; j < GRL_MAX_PARTS; ++j)
                    if (j < p.nparts) { sum += t[j][0]; sq += t[j][1]; }
                const float width = (float)(RL ? p.N : p.K), mean = sum / width;
                const float sd = sqrtf(fmaxf(sq / width - mean * mean, 0.f) + p.eps);
                *(f32x2_t*)(lds + VECS + bbuf * BIASB + 2 * COLB + 8 * tid) = f32x2_t{1.0f / sd, mean / sd};
            }
        }
    };

    for (;;) {
        const int npid = pid + (int)gridDim.x;
        const bool has_next = npid < ntiles;
        int m0n = 0, n0n = 0;
        if (has_next) {
            tile_of(npid, m0n, n0n);
            nextA = rsrc_of(p.A, m0n, p.M); nextW = rsrc_of(p.W, n0n, p.N);
            nextW2 = DUAL ? rsrc_of(p.W2, n0n, p.N) : nextW;
        } else nextA = nextW = nextW2 = make_rsrc_words(p.A, 0);      // transfers of a next tile that is not there: zeros, nothing is read

        // what every accumulator block starts from: the bias of its columns (and the beta of the norm that the epilogue re-forms on the residual) when
        // the staged epilogue follows, else zeros (the direct epilogue adds the bias itself; the folded LayerNorm scales the sum before its bias)
        f32x4 c4[4];
        auto start_values = [&](auto iq) {                   // (TR: a phase has columns of its own)
            static_for<4>([&](auto ic) {
                constexpr int c = decltype(ic)::value + (TR ? 4 * decltype(iq)::value : 0), b = c / 2, half = c % 2;
                constexpr bool up = DUAL && b >= TNO;
                f32x4 v = {0.f, 0.f, 0.f, 0.f};
                if (!LN && staged) {
                    const char* bl = lds + VECS + bbuf * BIASB + (wn * WNO + (b % TNO) * 32 + 16 * half + 4 * lq) * 4;
                    if (up ? p.bias2 : p.bias) v = *(const f32x4*)(bl + (up ? BNO * 4 : 0));
                    if constexpr (RL) v += *(const f32x4*)(bl + COLB);
                }
                c4[decltype(ic)::value] = v;
            });
        };
        start_values(std::integral_constant<int, 0>{});

        Acc16<WM / 32, TR ? 4 : 2> blocks;
        auto& acc = blocks.v;
        u32x4 fy[4][2], fx[2][2][2];
        auto step = [&](auto ifirst, int kt) {
            constexpr bool FIRST = decltype(ifirst)::value;
            const char* s = lds + (gstep & 1) * STAGE;
            int lch[2];
#pragma unroll
            for (int sl = 0; sl < 2; ++sl) lch[sl] = l4 * 128 + (((4 * sl + lq) ^ lds_swz<8>(l4)) << 4);
            auto read_y = [&](int q) {
#pragma unroll
                for (int sl = 0; sl < 2; ++sl)
#pragma unroll
                    for (int y = 0; y < 4; ++y) fy[y][sl] = *(const u32x4*)(s + (TR ? wn : wm) * 8192 + lch[sl] + q * HALFB + y * 2048);
            };
            auto read_x = [&](int q) {
#pragma unroll
                for (int sl = 0; sl < 2; ++sl)
#pragma unroll
                    for (int x = 0; x < 2; ++x) fx[q][x][sl] = *(const u32x4*)(s + (TR ? wm : wn) * 4096 + lch[sl] + (2 + q) * HALFB + x * 2048);
            };
            auto mfmas = [&](auto iq) {
                constexpr int q = decltype(iq)::value;
                __builtin_amdgcn_s_setprio(1);
                // (in serpentine order: from one instruction to the next an operand stays, 0.5 to 1 % of the products that the power limit bounds)
                static_for<32>([&](auto it) {
                    constexpr int t = decltype(it)::value, sl = t / 16, y = t / 4 % 4, x = y & 1 ? 3 - t % 4 : t % 4;
                    f32x4& to = acc[TR ? x : 4 * q + y][TR ? 4 * q + y : x];
                    const u32x4 &weights = TR ? fy[y][sl] : fx[x / 2][x % 2][sl], &rows = TR ? fx[x / 2][x % 2][sl] : fy[y][sl];
                    to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, weights), __builtin_bit_cast(bf16x8, rows), FIRST && sl == 0 ? c4[TR ? y : x] : to, 0, 0, 0);
                });
                __builtin_amdgcn_s_setprio(0);
            };
            auto reads_back = [&] {          // the reads of a memory part are back, everybody's behind the barrier
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            };
            auto meet = [&] {
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("s_barrier" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            };
            auto due = [&] {                 // everything but the last eight transfers (and the stores in front of them) has landed
                if (FIRST && stores_behind) wait_vmcnt<8 + STORES>();
                else wait_vmcnt<8>();
            };
            read_x(0); read_y(0); read_x(1);
            if (!FIRST && kt == 1 && has_next) issue_vectors(m0n, n0n, bbuf ^ 1);
            if constexpr (ASKS) if (kt == KT - 2 && staged) ask_for_residual();
            issue_half(H_Y1{}, gstep + 1);
            advance();
            due();                           // A1 of this step
            reads_back(); mfmas(std::integral_constant<int, 0>{}); meet();
            read_y(1);
            if constexpr (TR && FIRST) start_values(std::integral_constant<int, 1>{});
            issue_half(H_X0{}, gstep); issue_half(H_Y0{}, gstep); issue_half(H_X1{}, gstep);
            due();                           // B0, A0 and B1 of the next step
            if constexpr (FIRST) {
                merge_parts();
                if (RL && sums_due) finish_rows(m0p, n0p);
            }
            reads_back(); mfmas(std::integral_constant<int, 1>{});
            ++gstep;
        };
        step(std::true_type{}, 0);
        for (int kt = 1; kt < KT; ++kt) {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            step(std::false_type{}, kt);
        }
        // the waves in front meet the others' last matrix part here and run their epilogue beside it; the others meet them behind theirs
        __builtin_amdgcn_sched_barrier(0);
        if (!behind) asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);

        if (staged) {
            // EPI_ROPE: the lane's coordinates are formed anew; addresses kept over the tile loop spilled, and their reloads drained the transfers
            const int lane = EPI == EPI_ROPE ? fresh_lane() : tid & 63, l4 = lane & 15, lq = lane >> 4;
            char* own = lds + ((gstep - 1) & 1) * STAGE + HALFB + wave * 2048;
            const char* vec = lds + VECS + bbuf * BIASB;
            // this lane's 16-byte piece of a staged row: chunk cc of row rr (+ 2 per further read: a read's 8 rows are such that its turns meet no bank twice)
            const int cc = lane & (CB - 1), rr = CB == 8 ? ((lane >> 4) << 2) + ((lane >> 3) & 1) : lane >> 2;
            auto tile_rsrc = [&](const void* base) {
                const int64_t left = ((int64_t)(p.M - m0) * p.N - n0) * OES;
                return __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)base + ((int64_t)m0 * p.N + n0) * OES), 0, left > 0x7fffffff ? 0x7fffffff : (int)left, 0x00020000);
            };
            const __amdgpu_buffer_rsrc_t rsC = tile_rsrc(p.C), rsR = tile_rsrc(HASRES ? p.residual : p.C);
            constexpr int NONTEMPORAL = 2;
            int coff[GROUPS];
#pragma unroll
            for (int g = 0; g < GROUPS; ++g) {
                const int col = wn * WNO + g * UC + cc * EPCO;
                coff[g] = n0 + col < p.N ? (wm * WM + rr) * rowB + col * OES : (int)0x80000000;
            }
            // residual pieces: the memory counter retires in order, so all of them (bf16; fp32: a unit's, a unit ahead) are requested in front of the first store
            constexpr bool AT_ONCE = OES == 2;
            constexpr int AHEAD = AT_ONCE ? UNITS : 2;
            u32x4 res[HASRES ? AHEAD : 1][PER];
            auto fetch_res = [&](auto iu) {
                constexpr int u = decltype(iu)::value, i = u / GROUPS, g = u % GROUPS;
                if constexpr (HASRES) {
#pragma unroll
                    for (int j = 0; j < PER; ++j) res[u % AHEAD][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsR, coff[g], (16 * i + 2 * j) * rowB, NONTEMPORAL));
                }
            };
            float gq[RL ? GROUPS : 1][RL ? EPCO : 1];
            if constexpr (RL) static_for<GROUPS>([&](auto ig) {
                constexpr int g = decltype(ig)::value;
                const int nq = n0 + wn * WNO + g * UC + cc * EPCO;          // N is a multiple of the piece here
#pragma unroll
                for (int e = 0; e < EPCO; e += 4) {
                    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
                    const f32x4 gv = nq + e < p.N ? *(const f32x4*)(p.res_gamma + nq + e) : zero;
#pragma unroll
                    for (int k = 0; k < 4; ++k) gq[g][e + k] = gv[k];
                }
            });
            if constexpr (AT_ONCE) static_for<UNITS>([&](auto iu) { fetch_res(iu); });
            static_assert(!RL || (GROUPS == 2 && CB == 8), "a row's 16 pieces: 8 lanes, two units");
            float held[RL ? PER : 1][2];                      // RL: the sums of the first unit's pieces of a row
            // folded LayerNorm: sum_k LN(x)[m,k] W0[n,k] = rstd_m * acc[m,n] + (b'[n] - rstd_m * mean_m * c[n]), the vectors in registers
            f32x4 bv[LN ? 4 : 1], cv[LN ? 4 : 1];
            if constexpr (LN) static_for<4>([&](auto ic) {
                constexpr int b = decltype(ic)::value / 2, half = decltype(ic)::value % 2;
                constexpr bool up = DUAL && b >= TNO;
                const char* bl = vec + (wn * WNO + (b % TNO) * 32 + 16 * half + 4 * lq) * 4 + (up ? BNO * 4 : 0);
                bv[decltype(ic)::value] = (up ? p.bias2 : p.bias) ? *(const f32x4*)bl : f32x4{0.f, 0.f, 0.f, 0.f};
                cv[decltype(ic)::value] = *(const f32x4*)(bl + COLB);
            });
            static_assert(EPI != EPI_ROPE || (!DUAL && !LN && OES == 2), "a wave's 64 columns are one head");
            const bool rotated = EPI == EPI_ROPE && n0 + wn * WNO < p.rope_cols;
            // EPI_ROPE: the two halves of a pair, columns d and d + 32 of a head, are the same register of blocks b and b + 2, so the rotation
            // stays in registers: four multiply-adds a pair, on the sums before they are rounded.  cos and sin are requested a band ahead, the
            // bands' positions all at once (one by one, each waited for everything in flight).
            f32x4 cs[EPI == EPI_ROPE ? 2 : 1][2][2];
            int rope_at[EPI == EPI_ROPE ? WM / 16 : 1];           // where a row's values start in the table
            if constexpr (EPI == EPI_ROPE) if (rotated) {
                const int first = m0 + wm * WM + l4, last = p.M - 1;
                if (p.rope_pos) {
#pragma unroll
                    for (int i = 0; i < WM / 16; ++i) rope_at[i] = p.rope_pos[min(first + 16 * i, last)];
#pragma unroll
                    for (int i = 0; i < WM / 16; ++i) rope_at[i] = (int)min((uint32_t)rope_at[i], (uint32_t)(p.rope_S - 1));
                } else {
                    int turn = p.rope_S;
                    asm volatile("" : "+s"(turn));           // the divisor's reciprocal is formed here, not kept over the tile loop
#pragma unroll
                    for (int i = 0; i < WM / 16; ++i) rope_at[i] = min(first + 16 * i, last) % turn;
                }
#pragma unroll
                for (int i = 0; i < WM / 16; ++i) rope_at[i] = rope_at[i] * 64 + 8 * lq;
            }
            auto fetch_rope = [&](auto ii) {
                constexpr int i = decltype(ii)::value;
                if constexpr (EPI == EPI_ROPE) if (rotated) {
                    const float* t = (const float*)p.rope + rope_at[i];
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        cs[i & 1][b][0] = *(const f32x4*)(t + 32 * b);
                        cs[i & 1][b][1] = *(const f32x4*)(t + 32 * b + 4);
                    }
                }
            };
            fetch_rope(std::integral_constant<int, 0>{});
            // a unit: 16 rows of 64 or 128 bytes.  convert() writes it to this wave's place, collect() asks for it back, emit() stores it one unit later
            u32x4 val[2][PER];
            f32x2_t rst[2][RL ? PER : 1];
            auto convert = [&](auto iu) {
                constexpr int u = decltype(iu)::value, i = u / GROUPS, g = u % GROUPS;
                if constexpr (g == 0 && i + 1 < 8) fetch_rope(std::integral_constant<int, i + 1>{});
                if constexpr (!AT_ONCE) fetch_res(iu);
                float rs = 1.f, rm = 0.f;
                if constexpr (LN) {
                    const f32x2_t st = *(const f32x2_t*)(vec + 2 * COLB + 8 * (wm * WM + 16 * i + l4));
                    rs = st[0]; rm = st[1];
                }
                auto put = [&](int b, const float (&v)[4]) {          // four columns of block b of the unit
                    const int byte = (16 * b + 4 * lq) * OES;
                    store4<OutT>((OutT*)(own + l4 * UB + (((byte >> 4) ^ lds_swz<CB>(l4)) << 4) + (byte & 15)), v[0], v[1], v[2], v[3]);
                };
                if constexpr (EPI == EPI_ROPE) {
                    static_for<2>([&](auto ib) {
                        constexpr int b = decltype(ib)::value;
                        float v[4], w[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) { v[e] = acc[i][b][e]; w[e] = acc[i][b + 2][e]; }
                        if (rotated) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const float co = cs[i & 1][b][e >> 1][2 * (e & 1)], si = cs[i & 1][b][e >> 1][2 * (e & 1) + 1], x = v[e], y = w[e];
                                v[e] = x * co - y * si;
                                w[e] = y * co + x * si;
                            }
                        }
                        put(b, v);
                        put(b + 2, w);
                    });
                } else
                static_for<UC / 16>([&](auto ib) {
                    constexpr int b = g * (UC / 16) + decltype(ib)::value, b2 = DUAL ? b + 2 : b;
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = LN ? fmaf(acc[i][b][e], rs, fmaf(-rm, cv[LN ? b : 0][e], bv[LN ? b : 0][e])) : acc[i][b][e];
                    if constexpr (DUAL) {
                        float up[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) up[e] = LN ? fmaf(acc[i][b2][e], rs, fmaf(-rm, cv[LN ? b2 : 0][e], bv[LN ? b2 : 0][e])) : acc[i][b2][e];
                        glu_apply4(v, up, p);
                    } else if constexpr (EPI == EPI_GELU) gelu_fast4(v);
                    else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = epi_apply<EPI>(v[e], p);
                    }
                    put(decltype(ib)::value, v);
                });
            };
            // (a wave's LDS accesses are done in order: these reads see the unit's writes, and the next unit's writes come behind them)
            auto collect = [&](auto iu) {
                constexpr int u = decltype(iu)::value, i = u / GROUPS;
                asm volatile("" ::: "memory");
#pragma unroll
                for (int j = 0; j < PER; ++j) {
                    const int r = rr + 2 * j;
                    val[u & 1][j] = *(const u32x4*)(own + r * UB + ((cc ^ lds_swz<CB>(r)) << 4));
                    if constexpr (RL) rst[u & 1][j] = *(const f32x2_t*)(vec + 2 * COLB + 8 * (wm * WM + 16 * i + r));
                }
                asm volatile("" ::: "memory");
            };
            auto emit = [&](auto iu) {
                constexpr int u = decltype(iu)::value, i = u / GROUPS, g = u % GROUPS;
#pragma unroll
                for (int j = 0; j < PER; ++j) {
                    u32x4 out = val[u & 1][j];
                    if constexpr (EPI == EPI_RES) out = add_chunk<OutT>(out, res[u % AHEAD][j]);
                    if constexpr (RL) {
                        float xr[EPCO], o[EPCO];
                        Chunk<OutT>::unpack(res[u % AHEAD][j], xr);
                        Chunk<OutT>::unpack(out, o);
                        float sum = 0.f, sq = 0.f;
#pragma unroll
                        for (int e = 0; e < EPCO; ++e) o[e] = fmaf(fmaf(xr[e], rst[u & 1][j][0], -rst[u & 1][j][1]), gq[g][e], o[e]);
                        out = Chunk<OutT>::pack(o);
                        // (columns past N contribute 0: gamma, beta, bias and the products are 0 there)
                        Chunk<OutT>::moments(out, o, sum, sq);
                        if constexpr (g == 0) { held[j][0] = sum; held[j][1] = sq; }
                        else {
                            auto over_row = [](float a, float b) {          // piece c with c + 8, then + 4, + 2, + 1
                                float v = a + b;
                                v += dpp_move<0x1b>(dpp_move<0x141>(v));     // row_half_mirror, quad_perm 3,2,1,0: lane ^ 4
                                v += dpp_move<0x4e>(v);                      // quad_perm 2,3,0,1
                                return v + dpp_move<0xb1>(v);                // quad_perm 1,0,3,2
                            };
                            sum = over_row(held[j][0], sum); sq = over_row(held[j][1], sq);
                            if (cc == 0) *(f32x2_t*)(lds + SUMS_AT + wn * BM * 8 + 8 * (wm * WM + 16 * i + rr + 2 * j)) = f32x2_t{sum, sq};
                        }
                    }
                    // (the row's offset is added to the lane's, not passed as the scalar one: a VALU instruction right behind a four-word store may
                    // overwrite its data before the last lanes' is read; the compiler puts a wait state between them only where the scalar offset is
                    // zero, and without one elements came out wrong)
                    // written once, read by another kernel: keep it from displacing the operand panels in L2
                    __builtin_amdgcn_raw_buffer_store_b128(out, rsC, coff[g] + (16 * i + 2 * j) * rowB, 0, NONTEMPORAL);
                }
            };
            convert(std::integral_constant<int, 0>{});
            collect(std::integral_constant<int, 0>{});
            static_for<UNITS>([&](auto iu) {
                constexpr int u = decltype(iu)::value;
                if constexpr (u + 1 < UNITS) {
                    convert(std::integral_constant<int, u + 1>{});
                    collect(std::integral_constant<int, u + 1>{});
                }
                emit(iu);
            });
        } else if constexpr (!RL && EPI != EPI_ROPE) {        // EPI_RESLN and EPI_ROPE exist in the staged form only: the host launches them for nothing else
            epilogue_direct<OutT, 4, 2, TNO, WM, WNO, EPI, DUAL, LN>(blocks, p, m0, n0, wm, wn, lane);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (behind) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        stores_behind = staged;
        m0p = m0; n0p = n0; sums_due = true;
        if (!has_next) break;
        pid = npid; m0 = m0n; n0 = n0n; bbuf ^= 1;
    }
    if (!behind) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    finish_rows(m0p, n0p);
    wait_vmcnt<0>();                     // no transfer may be on its way to LDS that is somebody else's
}
