// Copies between the caller's arrays and the device.
//
// The caller's arrays are pageable, and the runtime's own copies of pageable memory go through one
// thread's staging: 38 GB/s in, 17 GB/s out on a link that carries 57 each way, and on a small
// call each waits for the host.  Here
//   * up to SMALL_COPY bytes pass through the context's pinned buffer: one memcpy and one
//     asynchronous copy per array;
//   * into the device, from there to CHUNKED_IN bytes, where one thread would move the chunks, the
//     runtime's copies are the fastest (MB: us, arrays used before / fresh ones; runtime, chunks): 4.5:
//     154 / 187, 179 / 214; 6: 195 / 241, 270 / 326; 8: 251 / 304, 304 / 367; 10: 297 / 365, 293 / 319;
//     12: 344 / 424, 386 / 415; 16: 450 / 568, 454 / 491; 24: 669 / 877, 613 / 636; 48: 1634 / 1663, 1114
//     / 1182 (a call with 12 MB from arrays used in turn: 3.57 ms by the runtime, 3.50 in chunks);
//   * larger ones, and what comes out of the device, are cut into chunks that several threads move
//     through pinned slots, each with a copy in flight while it touches the other slot's host side
//     (the page faults of a fresh result array spread over the threads too).  The slots and the streams are one set per device,
//     used by one transfer at a time.  A stream's first copies cost about 5 ms each (a process' first
//     84 MB in take 25 ms, 16 by the runtime, whose first 156 MB out take 16 against 4 here; the next
//     one or two in 7 instead of 2, with eight streams the next five), and two streams are slower
//     (18 MB out: 570 us, 480 with one per thread): four, which serve eight threads as well (84 MB in
//     1.9 ms, 397 MB out 9.7 ms, as with eight);
//   * where no pinned memory is to be had, the runtime copies.
// Particles in (MB: us) by the runtime / the pinned buffer / chunks: 0.11: 57 / 25 / 43; 1.9: 85 /
// 72 / 108; 3.8: 146 / 120 / 168; 7.7: 254 / 233 / 303; 214: 7814 / 9742 / 4290.  Out: 0.2: 128 / 50 / 98;
// 3.6: 213 / 206 / 191; 7.1: 1347 / 412 / 387; 14: 2549 / 794 / 459; 397: 39800 / 38200 / 9420.
// Four threads instead of eight: 397 out 10600; sixteen: 9400; chunks of 1 MB: 10900.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "transfer.h"
#include "vpmx_ctx.h"

namespace vpmx {

namespace {

constexpr size_t SMALL_COPY = 4 << 20, CHUNK = 2 << 20, PER_THREAD = 4 << 20, CHUNKED_IN = 2 * PER_THREAD;
constexpr int MAX_THREADS = 8, STREAMS = 4;

// The pinned slots (two per thread) and streams of one device.
struct Slots {
    std::mutex use;
    int device = 0;
    int ready = 0;  // threads whose slots are set up
    char *mem[MAX_THREADS] = {};
    hipStream_t stream[STREAMS] = {};  // thread t's: t mod STREAMS
    hipEvent_t done[MAX_THREADS][2] = {};
    // at least n threads' slots; the number there are (fewer when memory is short; what a thread
    // got before the call that failed stays for the next attempt)
    int grow(int n) {
        while (ready < n && set_up(ready)) ready++;
        if (ready < n) (void)hipGetLastError();  // (not an error of the transfer)
        return std::min(ready, n);
    }

private:
    bool set_up(int t) {
        void *p = nullptr;
        hipStream_t s;
        hipEvent_t e;
        if (!mem[t]) {
            if (hipHostMalloc(&p, 2 * CHUNK, hipHostMallocDefault) != hipSuccess) return false;
            mem[t] = (char *)p;
        }
        if (!stream[t % STREAMS]) {
            if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) return false;
            stream[t % STREAMS] = s;
        }
        for (hipEvent_t &d : done[t])
            if (!d) {
                if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
                d = e;
            }
        return true;
    }
};

// The device's slots, shared by its contexts and kept until the process ends (at most 32 MB pinned and
// the streams): memory, streams and first copies took 8 ms and taking them down 3 ms when a set had
// eight streams, more than a transfer of 200 MB saves, and a program that opens a context per
// evaluation paid it each time.
Slots &slots_of(int device) {
    static std::mutex m;
    static auto *all = new std::map<int, std::unique_ptr<Slots>>;  // (outlives the runtime's own shutdown)
    std::lock_guard<std::mutex> lock(m);
    std::unique_ptr<Slots> &s = (*all)[device];
    if (!s) {
        s.reset(new Slots());
        s->device = device;
    }
    return *s;
}

// Moves chunks (taken off `next`) through thread t's two slots.
hipError_t move_chunks(Slots &S, int t, bool in, const std::vector<Copy> &ch, std::atomic<size_t> &next) {
    const hipStream_t stream = S.stream[t % STREAMS];
    hipError_t e = hipSetDevice(S.device);
    const Copy *held[2] = {nullptr, nullptr};  // a slot's copy in flight
    // the slot's copy done: out, its bytes go to the caller
    auto settle = [&](int k) {
        if (!held[k] || e != hipSuccess) return;
        e = hipEventSynchronize(S.done[t][k]);
        if (e == hipSuccess && !in) std::memcpy(held[k]->dst, S.mem[t] + k * CHUNK, held[k]->bytes);
        held[k] = nullptr;
    };
    int k = 0;
    for (size_t i; e == hipSuccess && (i = next.fetch_add(1)) < ch.size(); k ^= 1) {
        settle(k);
        if (e != hipSuccess) break;
        char *slot = S.mem[t] + k * CHUNK;
        if (in) std::memcpy(slot, ch[i].src, ch[i].bytes);
        e = hipMemcpyAsync(in ? ch[i].dst : slot, in ? slot : ch[i].src, ch[i].bytes,
                           in ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipEventRecord(S.done[t][k], stream);
        held[k] = &ch[i];
    }
    settle(k);
    settle(k ^ 1);
    const hipError_t last = hipStreamSynchronize(stream);
    return e != hipSuccess ? e : last;
}

// The runtime's own copies.
int copy_direct(Ctx *c, bool in, const Copy *q, int n) {
    for (int i = 0; i < n; i++)
        if (q[i].bytes)
            VPMX_HIP(c, hipMemcpyAsync(q[i].dst, q[i].src, q[i].bytes,
                                       in ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, c->stream));
    VPMX_HIP(c, hipStreamSynchronize(c->stream));
    return VPMX_OK;
}

int copy_large(Ctx *c, bool in, const Copy *q, int n, size_t total) try {
    Slots &S = slots_of(c->device);
    std::vector<Copy> ch;
    for (int i = 0; i < n; i++)
        for (size_t o = 0; o < q[i].bytes; o += CHUNK)
            ch.push_back({(char *)q[i].dst + o, (const char *)q[i].src + o, std::min(CHUNK, q[i].bytes - o)});
    VPMX_HIP(c, hipStreamSynchronize(c->stream));  // what the copies read or overwrite
    std::lock_guard<std::mutex> lock(S.use);
    int nt = (int)std::min<size_t>(MAX_THREADS, total / PER_THREAD);
    const int cpus = (int)std::thread::hardware_concurrency();
    if (cpus > 0) nt = std::min(nt, cpus / 2);
    nt = S.grow(std::max(nt, 1));
    if (nt < 1) return copy_direct(c, in, q, n);
    std::atomic<size_t> next{0};
    hipError_t err[MAX_THREADS];
    std::fill(err, err + MAX_THREADS, hipSuccess);
    std::vector<std::thread> th;
    try {
        th.reserve((size_t)nt);
        for (int t = 1; t < nt; t++) th.emplace_back([&, t] { err[t] = move_chunks(S, t, in, ch, next); });
    } catch (...) {
        // no thread to be had: the ones there are take the chunks
    }
    err[0] = move_chunks(S, 0, in, ch, next);
    for (std::thread &t : th) t.join();
    for (hipError_t e : err) VPMX_HIP(c, e);
    return VPMX_OK;
} catch (const std::bad_alloc &) {  // (before the first copy)
    return copy_direct(c, in, q, n);
}

// The context's pinned buffer, no longer read by an earlier copy; null when there is no memory.
int small_buffer(Ctx *c, size_t bytes, char **out) {
    if (c->pin_busy) VPMX_HIP(c, hipStreamSynchronize(c->stream));
    c->pin_busy = false;
    if (c->pin_bytes < bytes) {
        if (c->pin) (void)hipHostFree(c->pin);
        c->pin = nullptr;
        c->pin_bytes = 0;
        if (hipHostMalloc(&c->pin, bytes + bytes / 4, hipHostMallocDefault) == hipSuccess) {
            c->pin_bytes = bytes + bytes / 4;
        } else {
            (void)hipGetLastError();
            c->pin = nullptr;
        }
    }
    *out = (char *)c->pin;
    return VPMX_OK;
}

size_t total_bytes(const Copy *q, int n) {
    size_t b = 0;
    for (int i = 0; i < n; i++) b += q[i].bytes;
    return b;
}

// A missing array is refused before any call of the runtime, whose last error would stay behind.
bool missing(const Copy *q, int n) {
    for (int i = 0; i < n; i++)
        if (q[i].bytes && (!q[i].src || !q[i].dst)) return true;
    return false;
}

// Result arrays that share memory: the runtime writes them one after another, so the last one's
// values stay (the threads of a large transfer would mix them).
bool shared_results(const Copy *q, int n) {
    for (int i = 0; i < n; i++)
        for (int j = 0; j < i; j++)
            if (q[i].bytes && q[j].bytes && (char *)q[i].dst < (char *)q[j].dst + q[j].bytes &&
                (char *)q[j].dst < (char *)q[i].dst + q[i].bytes)
                return true;
    return false;
}

// Memory that the device reaches by itself (pinned, managed, the device's own): the runtime
// copies it.
bool direct(const void *p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

bool any_direct(bool in, const Copy *q, int n) {
    for (int i = 0; i < n; i++)
        if (q[i].bytes && direct(in ? q[i].src : q[i].dst)) return true;
    return false;
}

}  // namespace

int copy_in(Ctx *c, const Copy *q, int n) {
    const size_t total = total_bytes(q, n);
    if (!total) return VPMX_OK;
    if (missing(q, n)) return fail(c, VPMX_ERR_HIP, "copy: invalid argument (a null array)");
    if ((total > SMALL_COPY && total < CHUNKED_IN) || any_direct(true, q, n)) return copy_direct(c, true, q, n);
    if (total > SMALL_COPY) return copy_large(c, true, q, n, total);
    char *b = nullptr;
    VPMX_TRY(small_buffer(c, total, &b));
    if (!b) return copy_direct(c, true, q, n);
    for (int i = 0; i < n; i++) {
        if (!q[i].bytes) continue;
        std::memcpy(b, q[i].src, q[i].bytes);
        c->pin_busy = true;
        VPMX_HIP(c, hipMemcpyAsync(q[i].dst, b, q[i].bytes, hipMemcpyHostToDevice, c->stream));
        b += q[i].bytes;
    }
    return VPMX_OK;
}

int copy_out(Ctx *c, const Copy *q, int n) {
    const size_t total = total_bytes(q, n);
    if (!total) return VPMX_OK;
    if (missing(q, n)) return fail(c, VPMX_ERR_HIP, "copy: invalid argument (a null array)");
    if (any_direct(false, q, n) || shared_results(q, n)) return copy_direct(c, false, q, n);
    if (total > SMALL_COPY) return copy_large(c, false, q, n, total);
    char *b = nullptr;
    VPMX_TRY(small_buffer(c, total, &b));
    if (!b) return copy_direct(c, false, q, n);
    c->pin_busy = true;
    char *p = b;
    for (int i = 0; i < n; i++) {
        if (q[i].bytes) VPMX_HIP(c, hipMemcpyAsync(p, q[i].src, q[i].bytes, hipMemcpyDeviceToHost, c->stream));
        p += q[i].bytes;
    }
    VPMX_HIP(c, hipStreamSynchronize(c->stream));
    c->pin_busy = false;
    p = b;
    for (int i = 0; i < n; i++) {
        if (q[i].bytes) std::memcpy(q[i].dst, p, q[i].bytes);
        p += q[i].bytes;
    }
    return VPMX_OK;
}

void free_transfer(Ctx *c) {
    if (c->pin) (void)hipHostFree(c->pin);
    c->pin = nullptr;
    c->pin_bytes = 0;
}

}  // namespace vpmx
