// host_copy.hip -- copies between pageable host memory and the device, through
// pinned buffers that several threads fill or empty.
//
// What bounds a pageable copy is the host's side of it: the link moves 64 MiB in
// 1.18 ms either way, one thread's memcpy takes 2.1 ms, four threads' 0.9 ms, and
// hipMemcpy on pageable memory 2.25 ms to the device and 3.9 ms back (256^3 FP32).
// Here a copy is cut into pieces that threads take in turn, each through one of
// kBuffers pinned buffers: while some are copied by the host, others are on the
// link.  The threads live for one copy (some 20 us each to start).  A host call of
// 10 steps at 256^3 FP32: 6.8 -> 4.0 ms.
#include "host_copy.h"

#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "api_common.h"

namespace perks {

namespace {

constexpr int kBuffers = kStagingBuffers;
constexpr int kThreads = 3;                     // with the caller's; 4 or 8, the same
constexpr size_t kMinStaged = (size_t)8 << 20;  // below, there is too little to overlap
constexpr int kMaxIdle = 2;  // sets kept between calls, until perks_release() (12 to 36 MiB each)

// Pinned buffers of one copy, and an event per buffer.
struct Staging {
    int dev = -1;
    size_t cap = 0;  // bytes of a buffer
    char* mem = nullptr;
    hipEvent_t ev[kBuffers] = {};

    bool create(size_t bytes)
    {
        cap = staging_capacity(bytes);
        if (hipGetDevice(&dev) != hipSuccess) return false;
        if (hipHostMalloc((void**)&mem, cap * kBuffers, hipHostMallocDefault) != hipSuccess) {
            mem = nullptr;
            return false;
        }
        for (hipEvent_t& e : ev) {
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                e = nullptr;
                return false;
            }
        }
        return true;
    }
    void destroy()
    {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        if (mem) (void)hipHostFree(mem);
    }
};

std::mutex g_mu;
std::vector<Staging*> g_idle;  // at most kMaxIdle

// First touch of new pinned pages costs some 0.4 ms a MiB, so a set outlives the
// call; concurrent calls each lease their own.
Staging* lease(size_t bytes)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        for (size_t i = 0; i < g_idle.size(); ++i) {
            if (g_idle[i]->dev != dev) continue;
            Staging* s = g_idle[i];
            g_idle.erase(g_idle.begin() + (long)i);
            return s;
        }
    }
    Staging* s = new (std::nothrow) Staging;
    if (s && !s->create(bytes)) {
        s->destroy();
        delete s;
        s = nullptr;
    }
    if (!s) (void)hipGetLastError();  // the caller takes the other way
    return s;
}

void give_back(Staging* s)
{
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if ((int)g_idle.size() < kMaxIdle) {
            try {
                g_idle.push_back(s);
                return;
            } catch (const std::bad_alloc&) {
            }
        }
    }
    s->destroy();
    delete s;
}

// Maps the whole pages of [p, p + bytes), as writing them would, while the link is
// still busy with them: an array that the caller has just allocated has none, and
// its first touch is then most of a copy's host side.  Their bytes stay as they
// are; where the system has no such call, the copy itself maps them.  10 steps at
// FP32 into a new array: 10 MiB 1.75 -> 1.41 ms, 24 MiB 2.90 -> 2.47, 36 MiB 3.97 ->
// 3.14, 64 MiB 6.40 -> 5.90; into one that is mapped, as before (64 MiB 3.7, 3.7).
void map_pages(char* p, size_t bytes)
{
#ifdef MADV_POPULATE_WRITE
    constexpr int populate_write = MADV_POPULATE_WRITE;
#else
    constexpr int populate_write = 23;  // Linux 5.14
#endif
    constexpr uintptr_t kPage = 4096;
    const uintptr_t first = ((uintptr_t)p + kPage - 1) / kPage * kPage;
    const uintptr_t end = ((uintptr_t)p + bytes) / kPage * kPage;
    if (first < end) (void)madvise((void*)first, end - first, populate_write);
}

// One copy in pieces.  Piece c uses buffer c % kBuffers once piece c - kBuffers
// has left it.  A piece is copied by the host in `slices`, one or a thread's share
// each: where a copy has three pieces, a thread for each would have the link wait
// for a whole third at one end.  Host calls of 10 steps FP32 at 16, 24 and 36 MiB,
// one slice a piece and three: 1.25, 1.76 and 2.72 ms; 1.10, 1.50 and 2.46.
// Threads take slices in order, so of the slices taken and not done the lowest
// never waits for one that nobody works on.
struct Copy {
    Staging* s;
    char* dev;
    char* host;
    size_t bytes;
    bool up;  // to the device
    size_t piece_bytes;
    long pieces;
    long slices;  // of a piece
    std::atomic<long> next{0};
    std::atomic<long> copied[kBuffers];  // slices of the piece in a buffer that the host has copied
    std::atomic<long> queued[kBuffers];  // pieces queued on the link so far, per buffer
    std::atomic<bool> failed{false};

    char* buffer(long c) const { return s->mem + (size_t)(c % kBuffers) * s->cap; }
    size_t size(long c) const { return std::min(piece_bytes, bytes - (size_t)c * piece_bytes); }

    // Queues piece c's transfer between its buffer and the device.
    bool queue(long c)
    {
        const int b = (int)(c % kBuffers);
        char* d = dev + (size_t)c * piece_bytes;
        const hipError_t e = up ? hipMemcpyAsync(d, buffer(c), size(c), hipMemcpyHostToDevice, nullptr)
                                : hipMemcpyAsync(buffer(c), d, size(c), hipMemcpyDeviceToHost, nullptr);
        if (e != hipSuccess || hipEventRecord(s->ev[b], nullptr) != hipSuccess) return false;
        queued[b].store(c / kBuffers + 1, std::memory_order_release);
        return true;
    }
    // Until piece c's transfer is queued and over.
    bool arrived(long c)
    {
        const int b = (int)(c % kBuffers);
        while (queued[b].load(std::memory_order_acquire) <= c / kBuffers) {
            if (failed.load(std::memory_order_relaxed)) return false;
            std::this_thread::yield();
        }
        return hipEventSynchronize(s->ev[b]) == hipSuccess;
    }
    // The host's copy of slice q of piece c; the last one of a piece passes the
    // buffer on to the link.
    bool slice(long c, long q)
    {
        const size_t share = (piece_bytes / (size_t)slices + 4095) / 4096 * 4096;
        const size_t from = std::min(size(c), (size_t)q * share);
        const size_t n = q + 1 < slices ? std::min(share, size(c) - from) : size(c) - from;
        char* h = host + (size_t)c * piece_bytes + from;
        char* b = buffer(c) + from;
        if (up) {
            if (c >= kBuffers && !arrived(c - kBuffers)) return false;
            std::memcpy(b, h, n);
        } else {
            map_pages(h, n);
            if (!arrived(c)) return false;
            std::memcpy(h, b, n);
        }
        std::atomic<long>& k = copied[c % kBuffers];
        if (k.fetch_add(1, std::memory_order_acq_rel) + 1 < slices) return true;
        k.store(0, std::memory_order_relaxed);
        if (up) return queue(c);
        return c + kBuffers >= pieces || queue(c + kBuffers);
    }
    void work()
    {
        if (hipSetDevice(s->dev) != hipSuccess) failed.store(true);
        for (;;) {
            const long u = next.fetch_add(1, std::memory_order_relaxed);
            if (u >= pieces * slices || failed.load(std::memory_order_relaxed)) return;
            if (!slice(u / slices, u % slices)) failed.store(true);
        }
    }
};

int staged(Staging* s, char* dev, char* host, size_t bytes, bool up)
{
    Copy c;
    c.s = s;
    c.dev = dev;
    c.host = host;
    c.bytes = bytes;
    c.up = up;
    c.piece_bytes = staging_piece(s->cap, bytes);
    c.pieces = (long)((bytes + c.piece_bytes - 1) / c.piece_bytes);
    c.slices = c.pieces <= kBuffers ? kThreads : 1;
    for (auto& q : c.queued) q.store(0);
    for (auto& k : c.copied) k.store(0);
    if (!up) {
        for (long i = 0; i < std::min<long>(kBuffers, c.pieces); ++i)
            if (!c.queue(i)) c.failed.store(true);
    }
    std::thread th[kThreads - 1];
    for (std::thread& t : th) {
        try {
            t = std::thread([&c] { c.work(); });
        } catch (const std::exception&) {
            break;  // fewer threads, the same pieces
        }
    }
    c.work();
    for (std::thread& t : th)
        if (t.joinable()) t.join();
    // the buffers are idle, and the data there, from here on
    if (hipStreamSynchronize(nullptr) != hipSuccess) c.failed.store(true);
    return c.failed.load() ? PERKS_ERR_HIP : PERKS_OK;
}

// Memory the runtime knows (pinned, managed) goes over the link as it is.
bool pageable(const void* p)
{
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return at.type == hipMemoryTypeUnregistered;
}

int copy(void* dev, void* host, size_t bytes, bool up)
{
    if (bytes >= kMinStaged && pageable(host)) {
        if (Staging* s = lease(bytes)) {
            const int rc = staged(s, (char*)dev, (char*)host, bytes, up);
            give_back(s);
            return rc;
        }
    }
    const hipError_t e = up ? hipMemcpy(dev, host, bytes, hipMemcpyHostToDevice)
                            : hipMemcpy(host, dev, bytes, hipMemcpyDeviceToHost);
    return e == hipSuccess ? PERKS_OK : PERKS_ERR_HIP;
}

}  // namespace

void release_host_copy()
{
    std::vector<Staging*> idle;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        idle.swap(g_idle);
    }
    for (Staging* s : idle) {
        s->destroy();
        delete s;
    }
}

int copy_to_device(void* dst, const void* src, size_t bytes) { return copy(dst, const_cast<void*>(src), bytes, true); }
int copy_to_host(void* dst, const void* src, size_t bytes) { return copy(const_cast<void*>(src), dst, bytes, false); }

}  // namespace perks
