// Operators called on host arrays (what backend.fnn.* and backend.attention.* are built on): copies in, kernels, copies out.
//
// Bound: PCIe (56.7 GB/s each way measured, 48 + 48 with both directions busy), for small calls the latencies of launch and
// wait (11 us for an empty kernel).  So:
//   * small calls (5 MiB in and out together) never touch the copy engines, whose hand-over to the compute queue costs 10 us
//     each way, and no events: inputs are copied into one pinned slab, from where a kernel per MiB fetches them while the next
//     are copied; results up to 64 KiB are written straight into the slab by the operator's kernel, larger ones by a copy kernel;
//   * large calls are cut into blocks of rows (sequences, for attention).  Blocks come in and are computed on the context's
//     stream and leave on a second one, so both directions of PCIe are busy at once.  They come in through a ring of pinned
//     chunks that a few host threads fill (hostcopy.cpp), and results leave through a second one that those threads empty.
//     bf16 operands are converted by those threads, so half the bytes cross PCIe.
#include "common.hpp"
#include "hostcopy.hpp"
#include <algorithm>
#include <atomic>
#include <cstring>
#include <functional>

namespace {

// Pinned slabs of small calls, and what counts as small.  us per fp32 call as a slab / through the rings, once the helper threads
// are awake: linear with 1 MiB of weights 2.5 MiB 113 / 140, 3.5 MiB 141 / 160, 4.5 MiB 168 / 189, 5.5 MiB 203 / 208; attention
// 3.5 MiB 138 / 159, 4.5 MiB 160 / 182, 5.5 MiB 189 / 202; linear with 256 columns 3.5 MiB 140 / 150, 5.5 MiB 198 / 196, 7.5 MiB
// 276 / 243: where the result is most of it, the rings overlap its copies and the slab does not.
constexpr size_t SLAB = 2u << 20, SLAB_MAX = 5u << 20;
constexpr size_t SLAB_PART = 1u << 20;               // of a slab's inputs, fetched by the device while the next are copied (512 KiB: 3 - 5 % slower)
// Rings of pinned chunks, 16 MiB per direction.  Chunks move by copy kernels: the copy engines need 10 us from one transfer
// to the next (1 MiB: 37 GB/s, 512 KiB with an event behind each: 19 GB/s), kernels 2 us.
constexpr size_t CHUNK = 2u << 20, SLOTS = 8;
constexpr size_t CHUNK_MIN = 256u << 10;
// Bytes moved per block of a large call: tying the two streams together costs 15 us a block, and a block of few sequences leaves
// CUs idle.  Half of it: attention 12 MiB 334 -> 420 us, 20 MiB 530 -> 683, linear with 256 columns 12 MiB 344 -> 361.  Up to
// 16 MiB there is one block: nothing but the host's own copies overlaps the transfers there.
constexpr size_t BLOCK = 8u << 20;
constexpr size_t PAST_CACHES = 4u << 20;             // results from this size on are copied to the caller past the caches (4, 8, 16 MiB: level or ahead)
constexpr size_t DIRECT = 64u << 10;                 // results up to this size are written into pinned memory by the operator's kernel
constexpr int MAXBLOCKS = 8;

}  // namespace

struct grl_hostpipe {
    std::atomic<bool> refused{false};    // pinned memory was refused once: what needs more of it runs on the runtime's own copies
    std::mutex mu;                       // one large call of a context at a time
    std::mutex slab_mu;
    struct slab { char* p; size_t cap; };
    std::vector<slab> slabs;             // free slabs of small calls (at most as many as calls have run at once)
    hipStream_t down = nullptr;
    char* ring_up = nullptr; char* ring_down = nullptr;
    hipEvent_t up_done[SLOTS] = {}, down_done[SLOTS] = {};
    bool up_busy[SLOTS] = {};
    size_t up_next = 0;
    hipEvent_t out[MAXBLOCKS] = {};
    bool ready = false;
};

grl_hostpipe* grl_hostpipe_create() { return new grl_hostpipe(); }

void grl_hostpipe_destroy(grl_hostpipe* h) {
    if (!h) return;
    for (auto& s : h->slabs) hipHostFree(s.p);
    if (h->down) { hipStreamSynchronize(h->down); hipStreamDestroy(h->down); }
    if (h->ring_up) hipHostFree(h->ring_up);
    if (h->ring_down) hipHostFree(h->ring_down);
    for (auto& e : h->up_done) if (e) hipEventDestroy(e);
    for (auto& e : h->down_done) if (e) hipEventDestroy(e);
    for (auto& e : h->out) if (e) hipEventDestroy(e);
    delete h;
}

// pinned memory, or nullptr where the driver refuses it (a limit of the container, a full host): that is no error
static char* pinned(grl_ctx* c, size_t bytes) {
    void* p = nullptr;
    if (c->hostpipe->refused) return nullptr;
    if (hipSetDevice(c->device) == hipSuccess && hipHostMalloc(&p, bytes, hipHostMallocDefault) == hipSuccess && p) return (char*)p;
    (void)hipGetLastError();
    c->hostpipe->refused = true;
    return nullptr;
}

// streams, rings and events of the large calls, on first use (under h->mu); h->ready stays false where pinned memory is refused
static int pipe_ready(grl_ctx* c, grl_hostpipe* h) {
    if (h->ready) return GRL_OK;
    if (!h->ring_up && !(h->ring_up = pinned(c, CHUNK * SLOTS))) return GRL_OK;
    if (!h->ring_down && !(h->ring_down = pinned(c, CHUNK * SLOTS))) return GRL_OK;
    if (!h->down) GRL_CHECK_HIP(hipStreamCreateWithFlags(&h->down, hipStreamNonBlocking));
    auto event = [](hipEvent_t& e) { return e ? hipSuccess : hipEventCreateWithFlags(&e, hipEventDisableTiming); };
    for (auto& e : h->up_done) GRL_CHECK_HIP(event(e));
    for (auto& e : h->down_done) GRL_CHECK_HIP(event(e));
    for (auto& e : h->out) GRL_CHECK_HIP(event(e));
    h->ready = true;
    return GRL_OK;
}

// Without pinned memory: the runtime's copies of pageable memory, one at a time and waited for.  n values (kind
// GRL_COPY_F32_BF16 / GRL_COPY_BF16_F32, converted through a buffer) or, for GRL_COPY_F32, n bytes.
static int plain_in(grl_ctx* c, int kind, void* dst, const void* src, size_t n) {
    std::vector<uint16_t> half;
    if (kind == GRL_COPY_F32_BF16) {
        half.resize(n);
        grl_host_copy(kind, half.data(), src, n);
        src = half.data();
        n *= 2;
    }
    GRL_CHECK_HIP(hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, c->stream));
    GRL_CHECK_HIP(hipStreamSynchronize(c->stream));
    return GRL_OK;
}
static int plain_out(grl_ctx* c, int kind, void* dst, const void* src, size_t n) {
    std::vector<uint16_t> half(kind == GRL_COPY_BF16_F32 ? n : 0);
    const bool widen = !half.empty();
    GRL_CHECK_HIP(hipMemcpyAsync(widen ? (void*)half.data() : dst, src, widen ? n * 2 : n, hipMemcpyDeviceToHost, c->stream));
    GRL_CHECK_HIP(hipStreamSynchronize(c->stream));
    if (widen) grl_host_copy(kind, dst, half.data(), n);
    return GRL_OK;
}

int grl_copy_chunk_launch(hipStream_t s, void* dst, const void* src, size_t bytes);

// `bytes` at dst on the device = n values of src, converted on the way (kind), chunk by chunk on stream s (under h->mu)
static int send(grl_hostpipe* h, hipStream_t s, int kind, void* dst, const void* src, size_t n, const std::function<int()>& meanwhile) {
    const size_t ed = kind == GRL_COPY_F32_BF16 ? 2 : 4, es = 4;
    // a transfer of a few chunks overlaps the host's copying better when the chunks are smaller
    const size_t chunk = std::min(CHUNK, std::max(CHUNK_MIN, (n * ed / 2 + 4095) / 4096 * 4096)) / ed;
    for (size_t at = 0; at < n; at += chunk) {
        const size_t m = std::min(chunk, n - at), slot = h->up_next;
        h->up_next = (slot + 1) % SLOTS;
        if (h->up_busy[slot]) GRL_CHECK_HIP(hipEventSynchronize(h->up_done[slot]));
        char* pin = h->ring_up + slot * CHUNK;
        grl_host_copy(kind, pin, (const char*)src + at * es, m);
        int rc = grl_copy_chunk_launch(s, (char*)dst + at * ed, pin, m * ed);
        if (rc) return rc;
        GRL_CHECK_HIP(hipEventRecord(h->up_done[slot], s));
        h->up_busy[slot] = true;
        if (meanwhile && (rc = meanwhile())) return rc;
    }
    return GRL_OK;
}

// Results on their way out: chunks are requested as far ahead as the ring has room, and copied to the caller in order (bf16
// widened by the host threads, so that half the bytes cross PCIe).
struct Outflow {
    grl_hostpipe* h; hipStream_t s;
    bool past;                            // copied to the caller past the caches
    struct Piece { int kind; char* dst; const char* src; size_t n; hipEvent_t after; };
    std::vector<Piece> pieces;
    size_t asked = 0, taken = 0;          // pieces requested from the device, pieces delivered
    void add(int kind, void* dst, const void* src, size_t n, hipEvent_t after) {
        const size_t es = kind == GRL_COPY_BF16_F32 ? 2 : 4, ed = 4;
        const size_t chunk = std::min(CHUNK, std::max(CHUNK_MIN, (n * es / 2 + 4095) / 4096 * 4096)) / es;
        for (size_t at = 0; at < n; at += chunk) {
            pieces.push_back({kind, (char*)dst + at * ed, (const char*)src + at * es, std::min(chunk, n - at), after});
            after = nullptr;              // one wait per block
        }
    }
    int pump(bool finish) {
        for (;;) {
            while (asked < pieces.size() && asked - taken < SLOTS) {
                const Piece& p = pieces[asked];
                if (p.after) GRL_CHECK_HIP(hipStreamWaitEvent(s, p.after, 0));
                int rc = grl_copy_chunk_launch(s, h->ring_down + (asked % SLOTS) * CHUNK, p.src, p.n * (p.kind == GRL_COPY_BF16_F32 ? 2 : 4));
                if (rc) return rc;
                GRL_CHECK_HIP(hipEventRecord(h->down_done[asked % SLOTS], s));
                ++asked;
            }
            if (taken == asked) return GRL_OK;
            const hipEvent_t e = h->down_done[taken % SLOTS];
            if (finish) GRL_CHECK_HIP(hipEventSynchronize(e));
            else {
                const hipError_t q = hipEventQuery(e);
                if (q == hipErrorNotReady) { (void)hipGetLastError(); return GRL_OK; }
                GRL_CHECK_HIP(q);
            }
            const Piece& p = pieces[taken];
            grl_host_copy(p.kind, p.dst, h->ring_down + (taken % SLOTS) * CHUNK, p.n, past);
            ++taken;
        }
    }
};

// ---- plain transfers of large arrays (grl_h2d / grl_d2h and their converting forms), on the context's stream
static int transfer_in(grl_ctx* c, int kind, void* dst, const void* src, size_t n) {
    grl_hostpipe* h = c->hostpipe;
    std::lock_guard<std::mutex> lk(h->mu);
    int rc = pipe_ready(c, h);
    if (rc) return rc;
    if (!h->ready) return plain_in(c, kind, dst, src, kind == GRL_COPY_F32 ? n * 4 : n);
    return send(h, c->stream, kind, dst, src, n, nullptr);
}
static int transfer_out(grl_ctx* c, int kind, void* dst, const void* src, size_t n) {
    grl_hostpipe* h = c->hostpipe;
    std::lock_guard<std::mutex> lk(h->mu);
    int rc = pipe_ready(c, h);
    if (rc) return rc;
    if (!h->ready) return plain_out(c, kind, dst, src, kind == GRL_COPY_F32 ? n * 4 : n);
    Outflow o{h, c->stream, n * 4 >= PAST_CACHES};
    o.add(kind, dst, src, n, nullptr);
    rc = o.pump(true);
    if (rc) hipStreamSynchronize(c->stream);        // nothing may still be writing into the ring
    return rc;
}

// the smallest free slab of at least `need` bytes, or a new one; p is nullptr where pinned memory is refused
static grl_hostpipe::slab take_slab(grl_ctx* c, size_t need) {
    grl_hostpipe* h = c->hostpipe;
    grl_hostpipe::slab s = {nullptr, SLAB};
    {
        std::lock_guard<std::mutex> lk(h->slab_mu);
        size_t best = h->slabs.size();
        for (size_t i = 0; i < h->slabs.size(); ++i)
            if (h->slabs[i].cap >= need && (best == h->slabs.size() || h->slabs[i].cap < h->slabs[best].cap)) best = i;
        if (best < h->slabs.size()) {
            s = h->slabs[best];
            h->slabs.erase(h->slabs.begin() + (long)best);
        }
    }
    std::lock_guard<std::mutex> pool(c->mu);          // a slab is a pool block too, as far as the statistics go
    if (s.p) { c->stats.hits++; return s; }
    c->stats.misses++;
    while (s.cap < need) s.cap *= 2;
    s.p = pinned(c, s.cap);
    return s;
}
static void give_slab(grl_ctx* c, grl_hostpipe::slab s) {
    std::lock_guard<std::mutex> lk(c->hostpipe->slab_mu);
    c->hostpipe->slabs.push_back(s);
}

int grl_copy_bytes_launch(grl_ctx* c, void* dst, const void* src, size_t bytes);
int grl_copy_segments_launch(grl_ctx* c, const grl_segments& g);
int grl_gemm_nt_act_block(grl_ctx* c, int dtype, int64_t rows, int64_t M, int64_t N, int64_t K, const void* A, const void* W, const float* bias,
                          void* C, int epilogue, float alpha, float beta);
int grl_glu_nt_block(grl_ctx* c, int dtype, int64_t rows, int64_t M, int64_t N, int64_t K, const void* x, const void* W_gate, const void* W_up,
                     const float* b_gate, const float* b_up, void* out, float* gate_cache, float* up_cache, int activation);

// Host -> device, small: converted or copied into the staging ring, from where a copy kernel fetches it like any other kernel
// of the stream (the copy engine would be faster from about 1 MiB on, but every hand-over to it and back costs 10 us).
// A full ring waits for the stream, i.e. for every kernel still reading from it.
constexpr size_t STAGE_RING = 4u << 20, SMALL_COPY = 256u << 10;
static int stage_in(grl_ctx* c, int kind, void* dst, const void* src, size_t bytes, size_t n) {
    std::lock_guard<std::mutex> lk(c->stage_mu);
    if (!c->stage) {
        if (!(c->stage = pinned(c, STAGE_RING))) return plain_in(c, kind, dst, src, kind == GRL_COPY_F32 ? bytes : n);
        c->stage_cap = STAGE_RING;
    }
    if (c->stage_off + bytes > c->stage_cap) {
        GRL_CHECK_HIP(hipStreamSynchronize(c->stream));
        c->stage_off = 0;
    }
    char* slot = c->stage + c->stage_off;
    if (kind == GRL_COPY_F32) memcpy(slot, src, bytes);
    else grl_host_copy(kind, slot, src, n);
    int rc = grl_copy_bytes_launch(c, dst, slot, bytes);
    c->stage_off += (bytes + 255) & ~(size_t)255;
    return rc;
}

// device -> host, small: a copy kernel writes into a pinned slab
static int slab_out(grl_ctx* c, int kind, void* dst, const void* src, size_t bytes, size_t n) {
    const auto slab = take_slab(c, bytes);
    if (!slab.p) return plain_out(c, kind, dst, src, kind == GRL_COPY_F32 ? bytes : n);
    int rc = grl_copy_bytes_launch(c, slab.p, src, bytes);
    const hipError_t e = hipStreamSynchronize(c->stream);
    if (!rc && e != hipSuccess) { grl_set_error("grl_d2h: %s", hipGetErrorString(e)); rc = GRL_ERR_HIP; }
    if (!rc) {
        if (kind == GRL_COPY_F32) memcpy(dst, slab.p, bytes);
        else grl_host_copy(kind, dst, slab.p, n);
    }
    give_slab(c, slab);
    return rc;
}

// Returns when the caller's buffer has been consumed; the transfer itself is ordered on the context stream like a kernel
// launch (work enqueued later on this context sees the data, grl_sync / grl_d2h wait for it).
extern "C" int grl_h2d(grl_ctx* c, void* dst, const void* src, size_t bytes) {
    GRL_REQUIRE(c && (bytes == 0 || (dst && src)), GRL_ERR_ARG, "grl_h2d: null argument");
    if (!bytes) return GRL_OK;
    if (bytes <= SMALL_COPY) return stage_in(c, GRL_COPY_F32, dst, src, bytes, 0);
    const size_t whole = bytes & ~(size_t)3;
    int rc = transfer_in(c, GRL_COPY_F32, dst, src, whole / 4);
    return rc || whole == bytes ? rc : stage_in(c, GRL_COPY_F32, (char*)dst + whole, (const char*)src + whole, bytes - whole, 0);
}

extern "C" int grl_d2h(grl_ctx* c, void* dst, const void* src, size_t bytes) {
    GRL_REQUIRE(c && (bytes == 0 || (dst && src)), GRL_ERR_ARG, "grl_d2h: null argument");
    if (!bytes) return GRL_OK;
    if (bytes <= SMALL_COPY) return slab_out(c, GRL_COPY_F32, dst, src, bytes, 0);
    const size_t whole = bytes & ~(size_t)3;
    int rc = transfer_out(c, GRL_COPY_F32, dst, src, whole / 4);
    return rc || whole == bytes ? rc : slab_out(c, GRL_COPY_F32, (char*)dst + whole, (const char*)src + whole, bytes - whole, 0);
}

extern "C" int grl_upload(grl_ctx* c, int dtype, int64_t n, const float* src, void* dst) {
    GRL_REQUIRE(c && grl_valid_dtype(dtype) && n >= 0 && (n == 0 || (src && dst)), GRL_ERR_ARG, "grl_upload: bad argument");
    if (n == 0) return GRL_OK;
    if (dtype == GRL_F32) return grl_h2d(c, dst, src, (size_t)n * 4);
    if ((size_t)n * 2 <= SMALL_COPY) return stage_in(c, GRL_COPY_F32_BF16, dst, src, (size_t)n * 2, (size_t)n);
    return transfer_in(c, GRL_COPY_F32_BF16, dst, src, (size_t)n);
}

extern "C" int grl_download(grl_ctx* c, int dtype, int64_t n, const void* src, float* dst) {
    GRL_REQUIRE(c && grl_valid_dtype(dtype) && n >= 0 && (n == 0 || (src && dst)), GRL_ERR_ARG, "grl_download: bad argument");
    if (n == 0) return GRL_OK;
    if (dtype == GRL_F32) return grl_d2h(c, dst, src, (size_t)n * 4);
    if ((size_t)n * 2 <= SMALL_COPY) return slab_out(c, GRL_COPY_BF16_F32, dst, src, (size_t)n * 2, (size_t)n);
    return transfer_out(c, GRL_COPY_BF16_F32, dst, src, (size_t)n);
}

// ---- operators on host arrays -----------------------------------------------------------------------------------
namespace {

struct HostArray {
    const float* in; float* out;      // one of the two
    int64_t n;                        // values in all
    int64_t per_unit;                 // values per row / sequence; 0: the whole array belongs to every block (weights)
    bool f32;                         // keeps 32 bits on the device whatever the storage type (biases, masks, caches)
};

// run_on_host without pinned memory: everything in, the whole operator, everything out
int run_plain(grl_ctx* c, int dtype, int64_t units, HostArray* arrays, int count, const std::function<int(int64_t, int64_t, void**)>& op) {
    void* dev[8] = {};
    auto half = [&](const HostArray& a) { return dtype == GRL_BF16 && !a.f32; };
    int rc = GRL_OK;
    for (int i = 0; i < count && !rc; ++i) {
        const HostArray& a = arrays[i];
        if (!a.in && !a.out) continue;
        dev[i] = grl_malloc(c, std::max<size_t>((size_t)a.n * (half(a) ? 2 : 4), 1));
        if (!dev[i]) rc = GRL_ERR_OOM;
        else if (a.in && a.n) rc = plain_in(c, half(a) ? GRL_COPY_F32_BF16 : GRL_COPY_F32, dev[i], a.in, (size_t)a.n * (half(a) ? 1 : 4));
    }
    if (!rc) rc = op(0, units, dev);
    for (int i = 0; i < count && !rc; ++i) {
        const HostArray& a = arrays[i];
        if (a.out && a.n) rc = plain_out(c, half(a) ? GRL_COPY_BF16_F32 : GRL_COPY_F32, a.out, dev[i], (size_t)a.n * (half(a) ? 1 : 4));
    }
    for (void* p : dev) grl_free(c, p);
    return rc;
}

// Runs op(first unit, units, device pointers of the arrays at `first unit`) over `units` rows (rows == true) or sequences.
int run_on_host(grl_ctx* c, int dtype, int64_t units, bool rows, HostArray* arrays, int count, const std::function<int(int64_t, int64_t, void**)>& op) {
    grl_hostpipe* h = c->hostpipe;
    auto dsize = [&](const HostArray& a) { return (size_t)a.n * (dtype == GRL_BF16 && !a.f32 ? 2 : 4); };
    auto pad = [](size_t b) { return (b + 255) & ~(size_t)255; };
    size_t ins = 0, outs = 0;
    for (int i = 0; i < count; ++i) (arrays[i].in ? ins : outs) += pad(dsize(arrays[i]));
    void* dev[8];
    GRL_REQUIRE(count <= 8, GRL_ERR_ARG, "run_on_host: too many arrays");

    const grl_host_calling calling;
    if (ins + outs <= SLAB_MAX) {
        const auto slab = take_slab(c, ins + outs);
        if (!slab.p) return run_plain(c, dtype, units, arrays, count, op);
        const bool direct = outs <= DIRECT;
        grl_segments seg, back;
        void* owned[8] = {};
        char* res[8] = {};
        int rc = GRL_OK;
        size_t at = 0, oat = ins, held = 0;
        // pieces that lie in the slab, on their way to the device
        auto fetch = [&]() {
            const int r = seg.count ? grl_copy_segments_launch(c, seg) : GRL_OK;
            seg.count = 0;
            held = 0;
            return r;
        };
        for (int i = 0; i < count && !rc; ++i) {
            const HostArray& a = arrays[i];
            if (a.in) {
                dev[i] = owned[i] = grl_malloc(c, dsize(a));          // (pool blocks are at least 256 bytes, in powers of two)
                if (!dev[i]) { rc = GRL_ERR_OOM; break; }
                const bool half = dtype == GRL_BF16 && !a.f32;
                const size_t es = half ? 2 : 4, part = SLAB_PART / es;
                for (size_t v = 0; v < (size_t)a.n && !rc; v += part) {
                    const size_t m = std::min(part, (size_t)a.n - v);
                    grl_host_copy(half ? GRL_COPY_F32_BF16 : GRL_COPY_F32, slab.p + at + v * es, a.in + v, m);
                    auto& s = seg.s[seg.count++];
                    s.src = slab.p + at + v * es; s.dst = (char*)dev[i] + v * es; s.bytes = (int64_t)(m * es);
                    if ((held += m * es) >= SLAB_PART || seg.count == 8) rc = fetch();
                }
                at += pad(dsize(a));
            } else if (a.out) {
                res[i] = slab.p + oat;
                dev[i] = direct ? res[i] : (owned[i] = grl_malloc(c, dsize(a)));
                if (!dev[i]) { rc = GRL_ERR_OOM; break; }
                if (!direct) { back.s[back.count].src = dev[i]; back.s[back.count].dst = res[i]; back.s[back.count++].bytes = (int64_t)dsize(a); }
                oat += pad(dsize(a));
            } else dev[i] = nullptr;
        }
        if (!rc) rc = fetch();
        if (!rc) rc = op(0, units, dev);
        if (!rc && back.count) rc = grl_copy_segments_launch(c, back);
        const hipError_t e = hipStreamSynchronize(c->stream);          // also on failure: kernels may still read the slab
        if (!rc && e != hipSuccess) { grl_set_error("operator on host arrays: %s", hipGetErrorString(e)); rc = GRL_ERR_HIP; }
        for (int i = 0; i < count && !rc; ++i)
            if (arrays[i].out)
                grl_host_copy(dtype == GRL_BF16 && !arrays[i].f32 ? GRL_COPY_BF16_F32 : GRL_COPY_F32, arrays[i].out, res[i], (size_t)arrays[i].n,
                              (size_t)arrays[i].n * 4 >= PAST_CACHES);
        for (void* p : owned) grl_free(c, p);
        give_slab(c, slab);
        return rc;
    }

    std::lock_guard<std::mutex> lk(h->mu);
    int rc = pipe_ready(c, h);
    if (rc) return rc;
    if (!h->ready) return run_plain(c, dtype, units, arrays, count, op);
    // from two blocks on, transfers in, work and transfers out overlap
    size_t moving = 0;
    for (int i = 0; i < count; ++i) if (arrays[i].per_unit) moving += dsize(arrays[i]);
    int64_t blocks = std::min<int64_t>(std::min<int64_t>(MAXBLOCKS, (int64_t)(moving / BLOCK)), units);
    if (blocks < 1) blocks = 1;
    // rows: whole tiles where there are plenty, and always whole 16-byte units at a block's start (the kernels' fast paths)
    int64_t step = (units + blocks - 1) / blocks;
    if (rows) step = step > 256 ? (step + 255) / 256 * 256 : (step + 15) / 16 * 16;

    std::vector<void*> owned;
    size_t results = 0;
    for (int i = 0; i < count; ++i) if (arrays[i].out) results += (size_t)arrays[i].n * 4;
    Outflow o{h, h->down, results >= PAST_CACHES};
    auto body = [&]() -> int {
        for (int i = 0; i < count; ++i) {
            dev[i] = nullptr;
            if (!arrays[i].in && !arrays[i].out) continue;
            dev[i] = grl_malloc(c, std::max<size_t>(dsize(arrays[i]), 1));
            if (!dev[i]) return GRL_ERR_OOM;
            owned.push_back(dev[i]);
        }
        auto meanwhile = [&]() { return o.pump(false); };
        auto send_part = [&](int i, int64_t first, int64_t n) {
            const bool half = dtype == GRL_BF16 && !arrays[i].f32;
            return send(h, c->stream, half ? GRL_COPY_F32_BF16 : GRL_COPY_F32, (char*)dev[i] + first * (half ? 2 : 4), arrays[i].in + first, (size_t)n, meanwhile);
        };
        for (int i = 0; i < count; ++i)
            if (arrays[i].in && !arrays[i].per_unit) { int r = send_part(i, 0, arrays[i].n); if (r) return r; }
        int b = 0;
        for (int64_t u = 0; u < units; u += step, ++b) {
            const int64_t m = std::min(step, units - u);
            void* part[8];
            for (int i = 0; i < count; ++i) {
                const HostArray& a = arrays[i];
                const bool half = dtype == GRL_BF16 && !a.f32;
                part[i] = dev[i] ? (char*)dev[i] + u * a.per_unit * (half ? 2 : 4) : nullptr;
                if (a.in && a.per_unit) { int r = send_part(i, u * a.per_unit, m * a.per_unit); if (r) return r; }
            }
            int r = op(u, m, part);
            if (r) return r;
            GRL_CHECK_HIP(hipEventRecord(h->out[b], c->stream));
            for (int i = 0; i < count; ++i) {
                const HostArray& a = arrays[i];
                if (a.out) o.add(dtype == GRL_BF16 && !a.f32 ? GRL_COPY_BF16_F32 : GRL_COPY_F32, a.out + u * a.per_unit, part[i], (size_t)(m * a.per_unit), h->out[b]);
            }
            if ((r = o.pump(false))) return r;
        }
        return o.pump(true);
    };
    rc = body();
    if (rc) {       // leave nothing in flight: rings and device buffers are about to be used again
        hipStreamSynchronize(c->stream); hipStreamSynchronize(h->down);
    }
    for (void* p : owned) grl_free(c, p);
    return rc;
}

}  // namespace

static int check_host(const char* who, grl_ctx* c, int dtype, int64_t M, int64_t N, int64_t K) {
    GRL_REQUIRE(c, GRL_ERR_ARG, "%s: null context", who);
    GRL_REQUIRE(grl_valid_dtype(dtype), GRL_ERR_ARG, "%s: bad dtype %d", who, dtype);
    GRL_REQUIRE(M >= 0 && N >= 0 && K >= 0, GRL_ERR_SHAPE, "%s: negative dimension", who);
    GRL_REQUIRE(M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31), GRL_ERR_SHAPE, "%s: dimension exceeds 2^31-1", who);
    return GRL_OK;
}

extern "C" int grl_host_linear(grl_ctx* c, int dtype, int64_t M, int64_t N, int64_t K, const float* x, const float* W, const float* bias,
                               float* y, int epilogue, float alpha, float beta) {
    int rc = check_host("grl_host_linear", c, dtype, M, N, K);
    if (rc || M == 0 || N == 0) return rc;
    GRL_REQUIRE(y && (K == 0 || (x && W)), GRL_ERR_ARG, "grl_host_linear: null argument");
    HostArray a[4] = {{K ? W : nullptr, nullptr, N * K, 0, false}, {bias, nullptr, N, 0, true}, {K ? x : nullptr, nullptr, M * K, K, false},
                      {nullptr, y, M * N, N, false}};
    if (!bias) a[1].n = 0;
    return run_on_host(c, dtype, M, true, a, 4, [&](int64_t, int64_t m, void** d) {
        if (m < M) return grl_gemm_nt_act_block(c, dtype, M, m, N, K, d[2], d[0], (const float*)d[1], d[3], epilogue, alpha, beta);
        return grl_gemm_nt_act(c, dtype, dtype, m, N, K, d[2], d[0], (const float*)d[1], d[3], epilogue, alpha, beta);
    });
}

extern "C" int grl_host_glu(grl_ctx* c, int dtype, int64_t M, int64_t N, int64_t K, const float* x, const float* W_gate, const float* W_up,
                            const float* b_gate, const float* b_up, float* out, float* gate_cache, float* up_cache, int activation) {
    int rc = check_host("grl_host_glu", c, dtype, M, N, K);
    if (rc || M == 0 || N == 0) return rc;
    GRL_REQUIRE(out && K > 0 && x && W_gate && W_up, GRL_ERR_ARG, "grl_host_glu: null argument or K == 0");
    const bool both = b_gate && b_up;
    HostArray a[8] = {{W_gate, nullptr, N * K, 0, false}, {W_up, nullptr, N * K, 0, false},
                      {both ? b_gate : nullptr, nullptr, both ? N : 0, 0, true}, {both ? b_up : nullptr, nullptr, both ? N : 0, 0, true},
                      {x, nullptr, M * K, K, false}, {nullptr, out, M * N, N, false},
                      {nullptr, gate_cache, gate_cache ? M * N : 0, N, true}, {nullptr, up_cache, up_cache ? M * N : 0, N, true}};
    return run_on_host(c, dtype, M, true, a, 8, [&](int64_t, int64_t m, void** d) {
        return grl_glu_nt_block(c, dtype, M, m, N, K, d[4], d[0], d[1], (const float*)d[2], (const float*)d[3], d[5], (float*)d[6], (float*)d[7], activation);
    });
}

extern "C" int grl_host_fa2(grl_ctx* c, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, const float* Q, const float* K, const float* V,
                            const float* mask, float* O, float scale, int causal, int rope, float rope_base, float rope_scaling) {
    GRL_REQUIRE(c, GRL_ERR_ARG, "grl_host_fa2: null context");
    GRL_REQUIRE(grl_valid_dtype(dtype), GRL_ERR_ARG, "grl_host_fa2: bad dtype %d", dtype);
    GRL_REQUIRE(B >= 0 && S >= 0 && H >= 0 && D >= 0 && B < 65536 && H < 65536 && S < (1LL << 24) && D < (1LL << 24), GRL_ERR_SHAPE, "grl_host_fa2: bad shape");
    if (B * S * H * D == 0)      // an empty batch, or a head dim the kernels refuse: their checks answer
        return grl_fa2_fwd(c, dtype, B, S, H, D, Q, K, V, mask, O, scale, causal, rope, rope_base, rope_scaling, nullptr);
    GRL_REQUIRE(Q && K && V && O, GRL_ERR_ARG, "grl_host_fa2: null argument");
    const int64_t per = S * H * D;
    HostArray a[5] = {{Q, nullptr, B * per, per, false}, {K, nullptr, B * per, per, false}, {V, nullptr, B * per, per, false},
                      {mask, nullptr, mask ? B * S : 0, S, true}, {nullptr, O, B * per, per, false}};
    return run_on_host(c, dtype, B, false, a, 5, [&](int64_t, int64_t b, void** d) {
        return grl_fa2_fwd(c, dtype, b, S, H, D, d[0], d[1], d[2], (const float*)d[3], d[4], scale, causal, rope, rope_base, rope_scaling, nullptr);
    });
}
