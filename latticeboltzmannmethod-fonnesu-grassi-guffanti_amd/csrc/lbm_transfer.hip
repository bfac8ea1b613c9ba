// Copies of whole states and fields between the device and pageable host
// memory (lbm_transfer.h).
//
// The runtime's own path copies pageable memory through one thread: 10 GB/s
// into memory touched for the first time (a fresh array's pages are zeroed on
// the way), 17 GB/s otherwise, 30 GB/s from the host, against 57 GB/s for
// page-locked memory over this link.  Here kLanes threads each own a
// page-locked chunk and take every kLanes-th chunk of the copy: the link
// fills or drains one chunk while the other threads copy theirs.  97 MB
// down: 9.4 -> 2.9 ms; up: 3.2 -> 2.2 ms.
#include "lbm_transfer.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <thread>

namespace lbm {

namespace {

constexpr int kLanes = 6;
constexpr size_t kChunk = (size_t)2 << 20;
// Below, the threads' start costs what they save.  us, the runtime's path / the
// threads: down 6.5 MB 387 / 315, 72 MB 6750 / 2100; up 6.5 MB 225 / 310, 12.1 MB
// 460 / 475, 15.9 MB 583 / 572, 72 MB 2485 / 2005.
constexpr size_t kMinDown = (size_t)6 << 20, kMinUp = (size_t)15 << 20;

std::mutex g_refs_mu;
int g_refs = 0;
// The chunks; held for a whole copy.  A copy that finds them taken by
// another thread goes the runtime's way.
std::mutex g_lanes_mu;
char *g_chunks = nullptr;

// Whether the memory is pageable (unknown to the runtime).
bool pageable(const void *p)
{
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();  // unknown memory is no error of the caller's
        return true;
    }
    return at.type == hipMemoryTypeUnregistered;
}

hipError_t plain(void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t s)
{
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, s);
    return e != hipSuccess || kind == hipMemcpyHostToDevice ? e : hipStreamSynchronize(s);
}

// One lane's chunks of a copy.
hipError_t run_lane(int device, int lane, char *chunk, char *dst, const char *src, size_t bytes, hipMemcpyKind kind,
                    hipStream_t s)
{
    hipError_t e = hipSetDevice(device);
    hipEvent_t done = nullptr;
    if (e == hipSuccess) e = hipEventCreateWithFlags(&done, hipEventDisableTiming);
    for (size_t at = (size_t)lane * kChunk; at < bytes && e == hipSuccess; at += kLanes * kChunk) {
        const size_t n = std::min(kChunk, bytes - at);
        if (kind == hipMemcpyDeviceToHost) {
            e = hipMemcpyAsync(chunk, src + at, n, kind, s);
            if (e == hipSuccess) e = hipEventRecord(done, s);
            if (e == hipSuccess) e = hipEventSynchronize(done);
            if (e == hipSuccess) std::memcpy(dst + at, chunk, n);
        } else {
            std::memcpy(chunk, src + at, n);
            e = hipMemcpyAsync(dst + at, chunk, n, kind, s);
            if (e == hipSuccess) e = hipEventRecord(done, s);
            if (e == hipSuccess) e = hipEventSynchronize(done);
        }
    }
    if (done) (void)hipEventDestroy(done);
    return e;
}

hipError_t copy(int device, void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t s, bool soon)
{
    const void *host = kind == hipMemcpyDeviceToHost ? dst : src;
    if (bytes < (kind == hipMemcpyDeviceToHost ? kMinDown : kMinUp) || !pageable(host)) return plain(dst, src, bytes, kind, s);
    std::unique_lock<std::mutex> lanes(g_lanes_mu, std::try_to_lock);
    if (!lanes.owns_lock()) return plain(dst, src, bytes, kind, s);
    if (!g_chunks) {
        void *p = nullptr;
        if (hipHostMalloc(&p, kLanes * kChunk, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return plain(dst, src, bytes, kind, s);
        }
        g_chunks = (char *)p;
    }
    // The steps queued before the copy are waited for here, by this thread
    // alone: a run of many steps would otherwise hold every lane for its length.
    // Short work is left to the lanes, whose start it hides (10 us).
    if (!soon)
        if (const hipError_t e = hipStreamSynchronize(s); e != hipSuccess) return e;
    hipError_t res[kLanes];
    std::thread threads[kLanes];
    auto lane = [&](int k) {
        res[k] = run_lane(device, k, g_chunks + (size_t)k * kChunk, (char *)dst, (const char *)src, bytes, kind, s);
    };
    int started = 1;  // lane 0 and the lanes without a thread run here
    try {
        for (; started < kLanes; ++started) threads[started] = std::thread(lane, started);
    } catch (...) {
    }
    lane(0);
    for (int k = started; k < kLanes; ++k) lane(k);
    for (int k = 1; k < started; ++k) threads[k].join();
    // A lane that failed may have left its chunk, or its caller's memory, to
    // a copy in flight: all of them end before the chunks are given back.
    const hipError_t end = hipStreamSynchronize(s);
    for (const hipError_t e : res)
        if (e != hipSuccess) return e;
    return end;
}

}  // namespace

hipError_t copy_to_host(int device, void *dst, const void *src, size_t bytes, hipStream_t s, bool soon)
{
    return copy(device, dst, src, bytes, hipMemcpyDeviceToHost, s, soon);
}

hipError_t copy_to_device(int device, void *dst, const void *src, size_t bytes, hipStream_t s)
{
    return copy(device, dst, src, bytes, hipMemcpyHostToDevice, s, false);
}

namespace {

// Where the device sees one byte of page-locked host memory.
char *device_byte(const char *host)
{
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, host) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return at.type == hipMemoryTypeHost ? (char *)at.devicePointer : nullptr;
}

}  // namespace

void *device_view(const void *host, size_t bytes)
{
    // Only a part of the caller's memory may be page-locked (hipHostRegister):
    // a kernel that wrote past it would fault, where a copy is an error.
    char *first = device_byte((const char *)host);
    if (!first || bytes == 0) return first;
    return device_byte((const char *)host + bytes - 1) == first + bytes - 1 ? first : nullptr;
}

void transfer_retain()
{
    std::lock_guard<std::mutex> lock(g_refs_mu);
    ++g_refs;
}

void transfer_release()
{
    std::lock_guard<std::mutex> lock(g_refs_mu);
    if (--g_refs > 0) return;
    std::lock_guard<std::mutex> lanes(g_lanes_mu);
    if (g_chunks) (void)hipHostFree(g_chunks);
    g_chunks = nullptr;
}

}  // namespace lbm
