// Runs copy_to_host on the CPU runtime of hip/hip_runtime.h; `check CASE` exits
// with 0 when the case holds and prints what does not.
#include "lbm_hostcopy.h"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <thread>
#include <vector>

namespace {
thread_local hipError_t t_last = hipSuccess;
thread_local int t_dev = 0;
std::atomic<int> events{0}, buffers{0}, direct{0}, staged{0};
std::atomic<int> buffers_allowed{1 << 20}, events_allowed{1 << 20};
const void* pinned = nullptr;      // memory that the runtime knows
bool refuses_unknown = false;      // whether asking for other memory's attributes is an error
std::atomic<int> news_allowed{1 << 30};   // the next allocations by new; then one throws

hipError_t res(hipError_t e) {
    if (e != hipSuccess) t_last = e;
    return e;
}
}  // namespace

void* operator new(size_t n) {
    if (news_allowed-- == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

hipError_t hipGetLastError() {
    const hipError_t e = t_last;
    t_last = hipSuccess;
    return e;
}
hipError_t hipGetDevice(int* dev) { *dev = t_dev; return hipSuccess; }
hipError_t hipSetDevice(int dev) { t_dev = dev; return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    if (buffers >= buffers_allowed) return res(hipErrorOutOfMemory);
    *p = std::malloc(bytes);
    ++buffers;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { std::free(p); --buffers; return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    a->type = p == pinned ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return res(p != pinned && refuses_unknown ? hipErrorInvalidValue : hipSuccess);
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (events >= events_allowed) return res(hipErrorOutOfMemory);
    *e = (FakeEvent*)std::malloc(sizeof(FakeEvent));
    (*e)->dev = t_dev;
    ++events;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); --events; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) { return res(e->dev == st->dev ? hipSuccess : hipErrorInvalidHandle); }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t) {
    std::memcpy(dst, src, bytes);
    ++(bytes > ((size_t)1 << 20) ? direct : staged);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }

namespace {
int bad = 0;
void want(bool ok, const char* what) {
    if (!ok) { std::printf("not so: %s\n", what); bad = 1; }
}

constexpr size_t kBytes = (size_t)40 << 20;
std::vector<char> src(kBytes), dst(kBytes);

// One copy of 40 MiB on device dev; whether every byte arrived.
bool copy(int dev) {
    FakeStream st{dev};
    std::memset(dst.data(), 0, kBytes);
    const lbm::OutCopy c = {dst.data(), src.data(), kBytes};
    const hipError_t e = lbm::copy_to_host(&c, 1, dev, &st);
    return e == hipSuccess && std::memcmp(dst.data(), src.data(), kBytes) == 0;
}

// A context of device 1 read by a thread whose current device is 0.
void device() {
    t_dev = 0;
    want(copy(1), "the copy of the other device's context succeeds");
    want(t_dev == 0, "the caller's current device is what it was");
    want((staged > 0 && direct == 0) || std::thread::hardware_concurrency() < 2, "it went through the staging buffers");
}

// Host memory that runs out at every allocation of the copy in turn: the fields
// arrive, and the next copy has the buffers it had before.
void memory() {
    want(copy(0), "the first copy succeeds");
    const int made = buffers;
    for (int k = 0; k < 200; ++k) {
        news_allowed = k;
        want(copy(0), "a copy without memory succeeds");
        const bool thrown = news_allowed < 0;
        news_allowed = 1 << 30;
        want(events == 0, "its events are destroyed");
        buffers_allowed = 0;   // what is idle has to do
        staged = direct = 0;
        want(copy(0) && (direct == 0 || made == 0), "its buffers are there for the next copy");
        buffers_allowed = 1 << 20;
        if (!thrown || bad) break;
    }
    want(buffers == made, "no buffer is made again");
}

// What runs out and is done without leaves no error behind for the thread's next
// launch to report.
void errors() {
    hipGetLastError();
    buffers_allowed = 0;
    want(copy(0), "a copy without pinned memory succeeds");
    want(hipGetLastError() == hipSuccess, "and leaves no error");
    buffers_allowed = 5;
    want(copy(0), "a copy with a part of the pinned memory succeeds");
    want(hipGetLastError() == hipSuccess, "and leaves no error");
    events_allowed = 3;
    want(copy(0), "a copy without events succeeds");
    want(hipGetLastError() == hipSuccess, "and leaves no error");
}

// Pinned memory of the caller takes the card's own copy, other memory the staging
// buffers, whichever way the runtime says that it does not know it.
void own_pinned() {
    pinned = dst.data();
    want(copy(0), "a copy into pinned memory succeeds");
    want(staged == 0 && direct == 1, "without the staging buffers");
    pinned = nullptr;
    for (bool refuses : {false, true}) {
        refuses_unknown = refuses;
        staged = direct = 0;
        want(copy(0), "a copy into other memory succeeds");
        want((staged > 0 && direct == 0) || std::thread::hardware_concurrency() < 2, "through the staging buffers");
        want(hipGetLastError() == hipSuccess, "and leaves no error");
    }
}
}  // namespace

int main(int argc, char** argv) {
    for (size_t i = 0; i < kBytes; ++i) src[i] = (char)(i * 2654435761u >> 13);
    lbm::host_staging_retain();
    const char* name = argc > 1 ? argv[1] : "";
    if (!std::strcmp(name, "device")) device();
    else if (!std::strcmp(name, "memory")) memory();
    else if (!std::strcmp(name, "errors")) errors();
    else if (!std::strcmp(name, "pinned")) own_pinned();
    else want(false, "a case of that name");
    want(events == 0, "every event is destroyed");
    lbm::host_staging_release();
    want(buffers == 0, "every buffer is freed with the last context");
    return bad;
}
