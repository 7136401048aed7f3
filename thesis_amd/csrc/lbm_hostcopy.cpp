// A field copy into pageable memory runs at one core's pace: the runtime stages it
// and its thread takes the page faults of the caller's fresh array (256^3, 537 MB:
// 54 ms, 10 GB/s).  Here a few threads share the copy, each with two pinned buffers:
// while the card fills one, the thread empties the other (537 MB: 17.5 ms, 31 GB/s,
// and no more with 12 threads; 67 MB 7.4 -> 2.8 ms, 32 MB 4.1 -> 1.7 ms).
#include "lbm_hostcopy.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace lbm {

namespace {

constexpr size_t kChunk = (size_t)1 << 20;   // bytes of a staging buffer
constexpr int kMaxThreads = 8;               // two buffers each: at most 16 MiB pinned in the process
// Bytes that make another thread worth its start.
constexpr size_t kPerThread = (size_t)2 << 20;

// Pinning 16 MiB takes 1.7 ms: copies below this use buffers that are there, or the
// runtime's path (16 MB: 0.9 ms, 2.3 ms, and 3.0 ms with buffers made for it).
constexpr size_t kMakeFrom = (size_t)24 << 20;

std::mutex g_mutex;
void* g_free[2 * kMaxThreads];               // idle staging buffers
int g_idle = 0, g_made = 0, g_holders = 0;

void drop_idle() {   // g_mutex held
    for (int i = 0; i < g_idle; ++i) (void)hipHostFree(g_free[i]);
    g_made -= g_idle;
    g_idle = 0;
}

// The buffers and events of one copy, given back on every way out; nothing here
// allocates host memory.
struct Staging {
    void* buf[2 * kMaxThreads];
    hipEvent_t ev[2 * kMaxThreads] = {};
    int n = 0;   // buffers held
    // Up to want buffers, idle ones and, when make is set, new ones (fewer when
    // others hold them).
    Staging(int want, bool make) {
        std::lock_guard<std::mutex> lock(g_mutex);
        while (n < want) {
            if (g_idle > 0) {
                buf[n++] = g_free[--g_idle];
                continue;
            }
            void* p = nullptr;
            if (!make || g_made >= 2 * kMaxThreads) break;
            if (hipHostMalloc(&p, kChunk, hipHostMallocPortable) != hipSuccess) {
                (void)hipGetLastError();
                break;
            }
            ++g_made;
            buf[n++] = p;
        }
    }
    ~Staging() {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        std::lock_guard<std::mutex> lock(g_mutex);
        for (int i = 0; i < n; ++i) g_free[g_idle++] = buf[i];
        if (g_holders == 0) drop_idle();
    }
    Staging(const Staging&) = delete;
    Staging& operator=(const Staging&) = delete;
};

hipError_t plain(const OutCopy* c, int n, hipStream_t st) {
    for (int i = 0; i < n; ++i) {
        const hipError_t e = hipMemcpyAsync(c[i].dst, c[i].src, c[i].bytes, hipMemcpyDeviceToHost, st);
        if (e != hipSuccess) return e;
    }
    return hipStreamSynchronize(st);
}

// Memory that the runtime knows (pinned by the caller): the card writes it itself,
// which beats staging and copying again (256^3, 537 MB: 9.4 / 17.3 ms; 28 MB 0.54 /
// 1.0 ms).
bool known(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();   // some runtimes refuse the question for other memory
    return false;
}

// Makes dev the calling thread's current device while it lives: a stream's events
// have to be of its device, and the caller's device is not this file's to change.
struct OnDevice {
    int was = -1;
    hipError_t e;
    explicit OnDevice(int dev) {
        int now = dev;
        e = hipGetDevice(&now);
        if (e == hipSuccess && now != dev && (e = hipSetDevice(dev)) == hipSuccess) was = now;
    }
    ~OnDevice() {
        if (was >= 0) (void)hipSetDevice(was);
    }
};

struct Piece {
    char* dst;
    const char* src;
    size_t bytes;
};

// One thread's share: pieces t, t + nt, ... through its two buffers.
hipError_t drain(const std::vector<Piece>& p, size_t t, size_t nt, void* const* buf, hipEvent_t* ev, hipStream_t st) {
    size_t flight[2] = {0, 0};
    bool busy[2] = {false, false};
    int k = 0;
    auto empty = [&](int b) {
        if (!busy[b]) return hipSuccess;
        const hipError_t e = hipEventSynchronize(ev[b]);
        if (e == hipSuccess) std::memcpy(p[flight[b]].dst, buf[b], p[flight[b]].bytes);
        busy[b] = false;
        return e;
    };
    hipError_t e = hipSuccess;
    for (size_t i = t; i < p.size() && e == hipSuccess; i += nt, k ^= 1) {
        if ((e = empty(k)) != hipSuccess) break;
        if ((e = hipMemcpyAsync(buf[k], p[i].src, p[i].bytes, hipMemcpyDeviceToHost, st)) != hipSuccess) break;
        flight[k] = i;
        busy[k] = true;   // from here the buffer may be written: it is waited for below in any case
        if ((e = hipEventRecord(ev[k], st)) != hipSuccess) { busy[k] = false; break; }
    }
    for (int j = 0; j < 2; ++j, k ^= 1) {
        const hipError_t r = empty(k);
        if (e == hipSuccess) e = r;
    }
    return e;
}

// The copies by up to `want` threads; false when nothing was started (no buffers,
// events or host memory for them), else e is the outcome.
//
// What fails here and is done without must not stay behind as the thread's last
// error: the next launch would report it as its own.
bool staged(const OutCopy* c, int n, int dev, hipStream_t st, int want, bool make, hipError_t& e) {
    try {
        const OnDevice on(dev);
        Staging s(2 * want, make);
        const int nt = s.n / 2;
        e = on.e;
        for (int i = 0; i < 2 * nt && e == hipSuccess; ++i) e = hipEventCreateWithFlags(&s.ev[i], hipEventDisableTiming);
        if (e != hipSuccess) (void)hipGetLastError();
        if (nt < 2 || e != hipSuccess) return false;
        std::vector<Piece> p;
        for (int i = 0; i < n; ++i)
            for (size_t o = 0; o < c[i].bytes; o += kChunk)
                p.push_back({(char*)c[i].dst + o, (const char*)c[i].src + o, std::min(kChunk, c[i].bytes - o)});
        std::atomic<int> err{(int)hipSuccess};
        auto work = [&](int t) {   // on the caller's thread and on new ones
            const OnDevice mine(dev);
            hipError_t r = mine.e;
            if (r == hipSuccess) r = drain(p, (size_t)t, (size_t)nt, &s.buf[2 * t], &s.ev[2 * t], st);
            if (r != hipSuccess) err = (int)r;
        };
        std::vector<std::thread> th;
        th.reserve((size_t)nt);
        int started = 1;
        try {
            for (; started < nt; ++started) th.emplace_back(work, started);
        } catch (...) {   // no more threads: this one takes their shares
        }
        work(0);
        for (int t = started; t < nt; ++t) work(t);
        for (auto& t : th) t.join();
        e = (hipError_t)err.load();
        if (e != hipSuccess) (void)hipStreamSynchronize(st);   // nothing in flight into the buffers
        return true;
    } catch (...) {
        return false;
    }
}

}  // namespace

hipError_t copy_to_host(const OutCopy* c, int n, int dev, hipStream_t st) {
    size_t total = 0;
    for (int i = 0; i < n; ++i) total += c[i].bytes;
    const int want = (int)std::min<size_t>({(size_t)kMaxThreads, total / kPerThread,
                                            (size_t)std::max(1u, std::thread::hardware_concurrency())});
    hipError_t e = hipSuccess;
    if (want >= 2 && std::none_of(c, c + n, [](const OutCopy& o) { return known(o.dst); }) &&
        staged(c, n, dev, st, want, total >= kMakeFrom, e)) return e;
    return plain(c, n, st);
}

void host_staging_retain() {
    std::lock_guard<std::mutex> lock(g_mutex);
    ++g_holders;
}

void host_staging_release() {
    std::lock_guard<std::mutex> lock(g_mutex);
    if (--g_holders == 0) drop_idle();
}

}  // namespace lbm
