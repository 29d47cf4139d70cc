// pk_transfer.hip -- device memory to ordinary host memory.
//
// The runtime copies to pageable memory at 18 GB/s at best: on MI355X 250 us for 4.2 MB, 510 us for 9.2 MB, 1020 us
// for 18.4 MB and 3.9 ms for 70 MB into pages in use, 680 us, 1.25 ms, 2.0 ms and 7.8 ms into fresh ones.  Here a
// small kernel writes the bytes into pinned memory chunk by chunk (the link takes 50 GB/s), and host threads move
// each chunk on while the next ones are under way: 140, 250 and 450 us and 1.6 ms into pages in use, 490, 530 and
// 800 us and 2.5 ms into fresh ones.  What bounds it there is the host's first touch, hence the extra threads for
// large copies.  The pinned memory is allocated by the first copy that needs it: 1 to 1.5 ms in the first contexts
// of a process, 0.1 ms later.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <new>
#include <thread>

#include "pk_internal.h"

namespace {

constexpr size_t SMALL_CHUNK = 512 << 10, LARGE_CHUNK = 1 << 20;
constexpr int SLOTS = 8;         // chunks in flight; 8 MB of pinned memory at most
constexpr int BLOCKS = 128;      // enough to fill the link (32 to 512 blocks time alike)
constexpr int HELPERS = 3;       // host threads besides the caller; one more brought nothing below 70 MB
// up to here the caller alone keeps up (4 MB: 138 us alone in 512 KB chunks, 141 us with helpers in 1 MB ones;
// 9.2 MB: 306 against 245 us)
constexpr size_t ALONE = 6 << 20;
// below this the runtime's copy is as fast (187 KB, 373 KB, 953 KB: 18, 25 and 50 us against 20, 28 and 50 here into
// pages in use, 19, 74 and 175 against 23, 78 and 182 into fresh ones; 1.1 MB: 72 against 52 and 260 against 200)
constexpr size_t DIRECT = 1 << 20;

template <class V>
__global__ void __launch_bounds__(256) k_copy_out(const V* __restrict__ src, V* __restrict__ dst, long n)
{
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) dst[i] = src[i];
}

template <class V>
void copy_out(hipStream_t stream, const char* src, char* dst, size_t bytes)
{
    const long n = (long)(bytes / sizeof(V));
    hipLaunchKernelGGL(k_copy_out<V>, dim3((unsigned)std::min<long>(BLOCKS, (n + 255) / 256)), dim3(256), 0, stream,
                       (const V*)src, (V*)dst, n);
}

}  // namespace

// pinned staging of one context: kept with it, grown on demand up to SLOTS large chunks, used by one copy at a time
struct pk_staging {
    std::mutex busy;
    char* ring = nullptr;
    size_t bytes = 0;
    hipEvent_t ev[SLOTS] = {};

    bool ready(size_t want)
    {
        if (bytes >= want) return true;
        if (ring) (void)hipHostFree(ring);
        ring = nullptr;
        bytes = 0;
        for (auto& e : ev)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                e = nullptr;
                return false;
            }
        if (hipHostMalloc((void**)&ring, want, hipHostMallocDefault) != hipSuccess) {
            ring = nullptr;
            return false;
        }
        bytes = want;
        return true;
    }

    ~pk_staging()
    {
        for (auto& e : ev)
            if (e) (void)hipEventDestroy(e);
        if (ring) (void)hipHostFree(ring);
    }
};

pk_staging* pk_staging_create() { return new (std::nothrow) pk_staging(); }
void pk_staging_destroy(pk_staging* s) { delete s; }

namespace {

// the context's device for a launch, and the caller's again after it
struct DeviceScope {
    int before = -1;
    explicit DeviceScope(int device)
    {
        if (hipGetDevice(&before) != hipSuccess || before == device || hipSetDevice(device) != hipSuccess) before = -1;
    }
    ~DeviceScope()
    {
        if (before >= 0) (void)hipSetDevice(before);
    }
};

}  // namespace

// host <- dev on the context's stream; returns when the bytes are there
int pk_copy_to_host(pk_ctx* c, void* host, const void* dev, size_t bytes)
{
    if (bytes == 0) return PK_OK;
    const size_t chunk = bytes <= ALONE ? SMALL_CHUNK : LARGE_CHUNK;
    const long nchunk = (long)((bytes + chunk - 1) / chunk);
    const int slots = (int)std::min<long>(SLOTS, nchunk);
    // memory that the device reaches by itself takes the runtime's copy, as do small copies and odd bytes
    hipPointerAttribute_t at;
    bool staged = bytes >= DIRECT && (((uintptr_t)dev | bytes) & 3) == 0;
    if (staged) {
        const hipError_t r = hipPointerGetAttributes(&at, host);
        if (r != hipSuccess) (void)hipGetLastError();
        staged = r != hipSuccess || at.type == hipMemoryTypeUnregistered;
    }
    DeviceScope scope(c->device);
    pk_staging& s = *c->staging;
    std::unique_lock<std::mutex> lock(s.busy, std::defer_lock);
    if (staged) {
        lock.lock();
        if (!s.ready(slots * chunk)) {
            (void)hipGetLastError();
            staged = false;
        }
    }
    if (!staged) {
        PK_HIP(c, hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, c->stream));
        PK_HIP(c, hipStreamSynchronize(c->stream));
        return PK_OK;
    }
    std::atomic<long> issued{0}, next{0}, emptied[SLOTS];
    std::atomic<int> failed{0};
    for (auto& e : emptied) e.store(0);
    // chunk i goes through slot i % slots once the chunk before it has left the slot
    auto issue = [&] {
        for (long i = issued.load(); i < nchunk && !failed.load(); i++) {
            const int k = (int)(i % slots);
            if (i >= slots && emptied[k].load(std::memory_order_acquire) != i - slots + 1) return;
            const size_t at0 = (size_t)i * chunk, len = std::min(chunk, bytes - at0);
            if ((((uintptr_t)dev | len) & 15) == 0)
                copy_out<uint4>(c->stream, (const char*)dev + at0, s.ring + k * chunk, len);
            else
                copy_out<uint32_t>(c->stream, (const char*)dev + at0, s.ring + k * chunk, len);
            hipError_t r = hipGetLastError();
            if (r == hipSuccess) r = hipEventRecord(s.ev[k], c->stream);
            if (r != hipSuccess) failed.store((int)r);
            issued.store(i + 1, std::memory_order_release);
        }
    };
    auto drain = [&](bool caller) {
        for (;;) {
            if (caller) issue();
            const long i = next.fetch_add(1);
            if (i >= nchunk) {
                while (caller && issued.load() < nchunk && !failed.load()) issue();    // the helpers' last chunks
                break;
            }
            const int k = (int)(i % slots);
            while (!failed.load() && issued.load(std::memory_order_acquire) <= i) {
                if (caller)
                    issue();
                else
                    std::this_thread::yield();
            }
            hipError_t r;
            while (!failed.load() && (r = hipEventQuery(s.ev[k])) != hipSuccess) {
                if (r != hipErrorNotReady) failed.store((int)r);
                if (!caller) std::this_thread::yield();
            }
            if (failed.load()) break;
            const size_t at0 = (size_t)i * chunk;
            std::memcpy((char*)host + at0, s.ring + k * chunk, std::min(chunk, bytes - at0));
            emptied[k].store(i + 1, std::memory_order_release);
        }
    };
    issue();
    // the work queued before the copy may take long: wait for it before the helpers start
    if (!failed.load()) {
        const hipError_t r = hipEventSynchronize(s.ev[0]);
        if (r != hipSuccess) failed.store((int)r);
    }
    std::thread helper[HELPERS];
    if (bytes > ALONE)
        try {
            for (auto& t : helper) t = std::thread(drain, false);
        } catch (...) {                // no more threads: the caller copies what is left
        }
    drain(true);
    for (auto& t : helper)
        if (t.joinable()) t.join();
    if (failed.load()) {
        (void)hipStreamSynchronize(c->stream);
        (void)hipGetLastError();
        PK_HIP(c, (hipError_t)failed.load());
    }
    return PK_OK;
}
