// Copies between numpy arrays and the pinned rings the transfers run through.
//
// One core moves 13 (into pages the process has not touched yet) to 28 GB/s, PCIe 56 GB/s each way: a single-threaded copy is
// what bounds a numpy -> numpy call.  A handful of helper threads take it to 50 ... 100 GB/s (measured on 48 MiB: 1 thread
// 27.8 / 13.3, 4 threads 87.9 / 38.6, 8 threads 119.6 / 51.5 GB/s into pinned / fresh memory).  Conversions to and from bf16
// ride along: half the bytes cross PCIe and no cast kernel runs.
#include "hostcopy.hpp"
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <sched.h>
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

constexpr int TOUCH = -1;

void copy_range(int kind, void* dst, const void* src, size_t a, size_t b) {
    if (kind == GRL_COPY_F32) memcpy((float*)dst + a, (const float*)src + a, (b - a) * sizeof(float));
    else if (kind == GRL_COPY_F32_BF16) to_bf16((uint16_t*)dst + a, (const uint32_t*)src + a, b - a);
    else if (kind == TOUCH) for (size_t i = a * 4; i < b * 4; i += 4096) ((volatile char*)dst)[i] = 0;
    else from_bf16((uint32_t*)dst + a, (const uint16_t*)src + a, b - a);
}

// A job is an array cut into pieces; whoever is free takes the next piece, the calling thread included.  Workers look for
// the next job for some 50 us before they go to sleep: the chunks of one large transfer follow each other that closely.
class Crew {
public:
    static Crew& get() { static Crew* c = new Crew(); return *c; }      // never destroyed: its threads sleep until the process ends
    void copy(int kind, void* dst, const void* src, size_t n) {
        constexpr size_t PIECE = 16 * 1024;                              // values
        // too small to share, a forked child (the threads stayed in the parent), or another thread's job is on: alone
        if (n < 4 * PIECE || workers_ == 0 || getpid() != pid_ || !turn_.try_lock()) { copy_range(kind, dst, src, 0, n); return; }
        const size_t pieces = (n + PIECE - 1) / PIECE;
        kind_ = kind; dst_ = dst; src_ = src; n_ = n; piece_ = PIECE;
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
        turn_.unlock();
    }

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
    void work() {
        for (size_t i; (i = next_.fetch_add(1, std::memory_order_relaxed)) < pieces_;) {
            const size_t a = i * piece_, b = a + piece_ < n_ ? a + piece_ : n_;
            copy_range(kind_, dst_, src_, a, b);
        }
    }
    void loop() {
        unsigned seen = 0;
        for (;;) {
            for (int spin = 0; job_.load() == seen && spin < 1000; ++spin) _mm_pause();
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
    std::atomic<int> inside_{0};
    std::atomic<bool> open_{false};
    size_t pieces_ = 0, n_ = 0, piece_ = 0;
    int kind_ = 0, workers_ = 0;
    void* dst_ = nullptr;
    const void* src_ = nullptr;
    pid_t pid_ = 0;
};

}  // namespace

void grl_host_touch(void* p, size_t bytes) { Crew::get().copy(TOUCH, p, p, bytes / 4); }
void grl_host_copy(int kind, void* dst, const void* src, size_t n) { Crew::get().copy(kind, dst, src, n); }
