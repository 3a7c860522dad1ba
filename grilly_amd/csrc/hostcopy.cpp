// Copies between numpy arrays and the pinned rings the transfers run through.
//
// One core moves 13 (into pages the process has not touched yet) to 28 GB/s, PCIe 56 GB/s each way: a single-threaded copy is
// what bounds a numpy -> numpy call.  A handful of helper threads take it to 50 ... 100 GB/s (measured on 48 MiB: 1 thread
// 27.8 / 13.3, 4 threads 87.9 / 38.6, 8 threads 119.6 / 51.5 GB/s into pinned / fresh memory).  Conversions to and from bf16
// ride along: half the bytes cross PCIe and no cast kernel runs.
#include "hostcopy.hpp"
#include "../../include/grilly_hip.h"
#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <map>
#include <mutex>
#include <pthread.h>
#include <sched.h>
#include <sys/mman.h>
#include <thread>
#include <unistd.h>
#include <immintrin.h>

namespace {

#define GRL_CLONES __attribute__((target_clones("avx512f", "avx2", "default")))

GRL_CLONES void to_bf16(uint16_t* __restrict d, const uint32_t* __restrict s, size_t n) {
    for (size_t i = 0; i < n; ++i) {
        const uint32_t u = s[i];
        const uint32_t r = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
        const uint32_t q = (u >> 16) | 0x40u;
        d[i] = (uint16_t)((u & 0x7fffffffu) > 0x7f800000u ? q : r);
    }
}
GRL_CLONES void from_bf16(uint32_t* __restrict d, const uint16_t* __restrict s, size_t n) {
    for (size_t i = 0; i < n; ++i) d[i] = (uint32_t)s[i] << 16;
}

// float results past the caches: a store that misses reads its line first, so a result much larger than they are costs three
// passes over memory the ordinary way and two this way (49 MiB into pages already mapped: 890 -> 600 us beside the transfers,
// widened from bf16 690 -> 420).
void stream(float* d, const float* s, size_t n) {
    size_t i = 0;
    for (; i < n && ((uintptr_t)(d + i) & 15u); ++i) d[i] = s[i];
    for (; i + 8 <= n; i += 8) {
        const __m128i a = _mm_loadu_si128((const __m128i*)(s + i)), b = _mm_loadu_si128((const __m128i*)(s + i + 4));
        _mm_stream_si128((__m128i*)(d + i), a);
        _mm_stream_si128((__m128i*)(d + i + 4), b);
    }
    for (; i < n; ++i) d[i] = s[i];
    _mm_sfence();
}
void stream(uint32_t* d, const uint16_t* s, size_t n) {
    const __m128i zero = _mm_setzero_si128();
    size_t i = 0;
    for (; i < n && ((uintptr_t)(d + i) & 15u); ++i) d[i] = (uint32_t)s[i] << 16;
    for (; i + 8 <= n; i += 8) {
        const __m128i a = _mm_loadu_si128((const __m128i*)(s + i));
        _mm_stream_si128((__m128i*)(d + i), _mm_unpacklo_epi16(zero, a));
        _mm_stream_si128((__m128i*)(d + i + 4), _mm_unpackhi_epi16(zero, a));
    }
    for (; i < n; ++i) d[i] = (uint32_t)s[i] << 16;
    _mm_sfence();
}

void copy_range(int kind, bool past, void* dst, const void* src, size_t a, size_t b) {
    if (past && kind == GRL_COPY_F32) { stream((float*)dst + a, (const float*)src + a, b - a); return; }
    if (past && kind == GRL_COPY_BF16_F32) { stream((uint32_t*)dst + a, (const uint16_t*)src + a, b - a); return; }
    if (kind == GRL_COPY_F32) memcpy((float*)dst + a, (const float*)src + a, (b - a) * sizeof(float));
    else if (kind == GRL_COPY_F32_BF16) to_bf16((uint16_t*)dst + a, (const uint32_t*)src + a, b - a);
    else from_bf16((uint32_t*)dst + a, (const uint16_t*)src + a, b - a);
}

// A job is an array cut into pieces; whoever is free takes the next piece, the calling thread included.  Workers look for
// the next job for some 20 us before they go to sleep, which is how closely the chunks of one transfer follow each other, and for
// some 200 us while an operator on host arrays is under way: its result is copied when the device is through.  (Asleep again by
// then: 512 rows of attention 2.5 MiB 110 -> 122 us, linear with 256 columns 4 MiB 155 -> 164.)
class Crew {
public:
    static Crew& get() { static Crew* c = new Crew(); return *c; }      // never destroyed: its threads sleep until the process ends
    void copy(int kind, void* dst, const void* src, size_t n, bool past) {
        constexpr size_t PIECE = 16 * 1024;                              // values
        // too small to share, a forked child (the threads stayed in the parent), or another thread's job is on: alone
        // or the CPUs have turned out to be taken
        const int64_t begin = now();
        if (n < 4 * PIECE || workers_ == 0 || begin < alone_until_.load(std::memory_order_relaxed) || getpid() != pid_ || !turn_.try_lock()) {
            copy_range(kind, past, dst, src, 0, n);
            return;
        }
        const size_t pieces = (n + PIECE - 1) / PIECE;
        kind_ = kind; past_ = past; dst_ = dst; src_ = src; n_ = n; piece_ = PIECE;
        next_.store(0, std::memory_order_relaxed);
        pieces_ = pieces;
        open_.store(true);
        {
            std::lock_guard<std::mutex> lk(mu_);
            job_.fetch_add(1);
        }
        cv_.notify_all();
        work();
        // No piece is left.  A worker that has entered the job may still be copying one; one that wakes up later finds the
        // job closed and touches nothing of it, so there is no waiting for sleepers.
        open_.store(false);
        while (inside_.load() != 0) _mm_pause();
        judge(begin, now(), n);
        turn_.unlock();
    }

    void call(int d) { calls_.fetch_add(d, std::memory_order_relaxed); }

private:
    Crew() {
        cpu_set_t set;
        CPU_ZERO(&set);
        int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
        pid_ = getpid();
        workers_ = cpus / 2 - 1;
        workers_ = workers_ < 0 ? 0 : workers_ > 7 ? 7 : workers_;
        for (int i = 0; i < workers_; ++i) std::thread([this] { loop(); }).detach();
    }
    static int64_t now() { return std::chrono::duration_cast<std::chrono::nanoseconds>(std::chrono::steady_clock::now().time_since_epoch()).count(); }
    // Where every CPU already runs a thread (the threads of a BLAS or an OpenMP runtime spin for 1 - 200 ms behind each of its calls),
    // helpers do harm: one that loses its CPU in the middle of a piece, or takes the caller's, holds the call up for time slices of
    // some milliseconds.  A job that takes far longer than its bytes is the sign of it.  After two of them within 20 ms the caller
    // copies alone for 20 ms, and twice as long each time it happens again soon after.  Mean us per call with a 1024-cube product of
    // numpy before each, always with helpers / with this: attention 32 x 64 x 8 x 64 1445 - 1840 / 540 - 660, in bf16
    // 1090 - 1560 / 390 - 480, fused_linear_gelu 4000 x 3072 x 768 3600 - 4500 / 2300 - 2600.
    void judge(int64_t begin, int64_t end, size_t n) {
        constexpr int64_t SLACK = 300000, FIRST = 20000000, LONGEST = 640000000;        // ns
        if (end - begin <= SLACK + (int64_t)n) return;                                  // 4 GB/s, a quarter of what one thread moves
        const bool soon = begin - alone_until_.load(std::memory_order_relaxed) < 2 * pause_, twice = begin - stalled_ < FIRST;
        stalled_ = end;
        if (!soon && !twice) return;
        pause_ = soon ? std::min(2 * pause_, LONGEST) : FIRST;
        alone_until_.store(end + pause_, std::memory_order_relaxed);
    }
    void work() {
        for (size_t i; (i = next_.fetch_add(1, std::memory_order_relaxed)) < pieces_;) {
            const size_t a = i * piece_, b = a + piece_ < n_ ? a + piece_ : n_;
            copy_range(kind_, past_, dst_, src_, a, b);
        }
    }
    void loop() {
        unsigned seen = 0;
        for (;;) {
            for (int spin = 0; job_.load() == seen && spin < (calls_.load(std::memory_order_relaxed) ? 10000 : 1000); ++spin)
                _mm_pause();
            if (job_.load() == seen) {
                std::unique_lock<std::mutex> lk(mu_);
                cv_.wait(lk, [&] { return job_.load() != seen; });
            }
            seen = job_.load();
            inside_.fetch_add(1);              // before the look at open_: the caller closes the job, then waits for inside_ == 0
            if (open_.load()) work();
            inside_.fetch_sub(1);
        }
    }
    std::mutex turn_, mu_;
    std::condition_variable cv_;
    std::atomic<unsigned> job_{0};
    std::atomic<size_t> next_{0};
    std::atomic<int> inside_{0}, calls_{0};
    std::atomic<bool> open_{false};
    std::atomic<int64_t> alone_until_{0};
    int64_t pause_ = 0, stalled_ = -1000000000;
    size_t pieces_ = 0, n_ = 0, piece_ = 0;
    int kind_ = 0, workers_ = 0;
    bool past_ = false;
    void* dst_ = nullptr;
    const void* src_ = nullptr;
    pid_t pid_ = 0;
};

// ---- memory for large results
// The C library maps every block above 32 MiB afresh and unmaps it when it is freed, so a result of that size pays a fault and
// the zeroing of every page: the 48 MiB result of a 4000 x 3072 x 768 product took 4.1 ms of numpy call in such memory, 1.7 ms
// in pages the process has already (24 MiB results: 0.60 ms both ways).  Freed blocks are kept here and handed out again, up
// to IDLE_MAX of them waiting.  They are ordinary private pages: a forked child has its own copy of them.
class Results {
public:
    static Results& get() { static Results* r = new Results(); return *r; }     // never destroyed: arrays may outlive everything else
    void* take(size_t bytes) {
        const size_t len = (std::max<size_t>(bytes, 1) + PAGE - 1) / PAGE * PAGE;
        if (len < bytes) return nullptr;
        std::lock_guard<std::mutex> lk(mu_);
        auto best = idle_.end();
        for (auto it = idle_.begin(); it != idle_.end(); ++it)
            if (it->second >= len && it->second <= len + len / 4 && (best == idle_.end() || it->second < best->second)) best = it;
        if (best != idle_.end()) {
            void* p = best->first;
            live_[p] = best->second;
            waiting_ -= best->second;
            idle_.erase(best);
            return p;
        }
        void* p = mmap(nullptr, len, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
        if (p == MAP_FAILED) return nullptr;
        madvise(p, len, MADV_HUGEPAGE);
        live_[p] = len;
        return p;
    }
    size_t size(void* p) {
        std::lock_guard<std::mutex> lk(mu_);
        auto it = live_.find(p);
        return it == live_.end() ? 0 : it->second;
    }
    void give(void* p) {
        std::lock_guard<std::mutex> lk(mu_);
        auto it = live_.find(p);
        if (it == live_.end()) return;
        const size_t len = it->second;
        live_.erase(it);
        drop_to(len > IDLE_MAX ? IDLE_MAX : IDLE_MAX - len);
        if (len > IDLE_MAX) { munmap(p, len); return; }
        idle_[p] = len;
        waiting_ += len;
    }
    void trim() {
        std::lock_guard<std::mutex> lk(mu_);
        drop_to(0);
    }

private:
    static constexpr size_t PAGE = 4096, IDLE_MAX = 512u << 20;
    // a child forked while another thread is in here would find the lock taken for ever
    Results() { pthread_atfork([] { get().mu_.lock(); }, [] { get().mu_.unlock(); }, [] { get().mu_.unlock(); }); }
    void drop_to(size_t most) {
        while (waiting_ > most) {
            munmap(idle_.begin()->first, idle_.begin()->second);
            waiting_ -= idle_.begin()->second;
            idle_.erase(idle_.begin());
        }
    }
    std::mutex mu_;
    std::map<void*, size_t> live_, idle_;
    size_t waiting_ = 0;
};

void* result_realloc(void*, void* p, size_t bytes) {
    const size_t old = p ? Results::get().size(p) : 0;
    if (p && bytes <= old && bytes >= old / 2) return p;
    void* q = Results::get().take(bytes);
    if (q && p) {
        memcpy(q, p, std::min(old, bytes));
        Results::get().give(p);
    }
    return q;
}
void* result_calloc(void*, size_t n, size_t each) {
    size_t bytes;
    if (__builtin_mul_overflow(n, each, &bytes)) return nullptr;
    void* p = Results::get().take(bytes);
    if (p) memset(p, 0, bytes);
    return p;
}

// numpy's public allocator interface, version 1: PyDataMem_Handler of numpy/ndarraytypes.h
struct NumpyHandler {
    char name[127];
    uint8_t version;
    struct {
        void* ctx;
        void* (*malloc)(void*, size_t);
        void* (*calloc)(void*, size_t, size_t);
        void* (*realloc)(void*, void*, size_t);
        void (*free)(void*, void*, size_t);
    } allocator;
};
const NumpyHandler numpy_handler = {"grilly_results", 1, {nullptr, [](void*, size_t n) { return Results::get().take(n); }, result_calloc, result_realloc,
                                                          [](void*, void* p, size_t) { if (p) Results::get().give(p); }}};

}  // namespace

void grl_host_copy(int kind, void* dst, const void* src, size_t n, bool past_caches) { Crew::get().copy(kind, dst, src, n, past_caches); }
void grl_host_call(int change) { Crew::get().call(change); }
void grl_host_trim() { Results::get().trim(); }

extern "C" void* grl_host_alloc(size_t bytes) { return bytes ? Results::get().take(bytes) : nullptr; }
extern "C" void grl_host_free(void* p) { if (p) Results::get().give(p); }
extern "C" const void* grl_numpy_handler(void) { return &numpy_handler; }
