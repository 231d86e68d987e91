// transfer.hip -- copies between the caller's (pageable) arrays and device
// memory through pinned slots, several host threads at a time.
//
// What bounds it: the PCIe link reaches 56 GB/s from and to pinned memory.  A
// plain copy to pageable memory reaches 18 GB/s (one thread copies out of the
// runtime's own staging buffer, behind it), and a first write to a fresh array
// adds the zeroing of its pages (30 GB/s): a 64 MiB density took 6 ms.  Here
// each thread has two slots, one in flight while it copies the other, so that
// the copies to the caller's pages and their faults run beside the link.
#include "kernels.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace t2 {

namespace {

constexpr size_t SLOT = 1ull << 21;      // bytes per slot
constexpr int WORKERS = 6;               // threads at most, the caller's among them
// below these one plain copy is as fast: a fresh array of 2.1 MB takes 163 us
// either way, 4.2 MB 316 -> 276, 8.4 MB 592 -> 466, 67 MB 6306 -> 1927; up, the
// plain copy reaches 38 GB/s and 6 MB are slower in pieces (446 -> 514 us a
// circumcenter call), 22 MB faster (1394 -> 1313)
constexpr size_t LEAST_DOWN = 3ull << 20, LEAST_UP = 1ull << 24;
// bytes that make another thread worth its start (4 MiB: 8.4 MB 592 us); slots
// of 1 MiB or 512 KiB pay more per copy (67 MB 2294, 3247 us)
constexpr size_t PER_WORKER = 1ull << 21;

// The slots of the process, two per worker: allocated by the first large
// copy, freed when the last context closes.  One copy uses them at a time;
// one that finds them taken goes the plain way.
struct Slots {
    std::mutex mu;
    unsigned char *base = nullptr;
    int users = 0;
};

Slots &slots()
{
    static Slots *s = new Slots;   // never destroyed: contexts may outlive static objects
    return *s;
}

struct Job {
    unsigned char *host, *dev;
    size_t bytes;
    bool up;               // host to device
    hipStream_t s;
    int device, workers;
    unsigned char *base;
    std::atomic<int> err{0};
};

// worker w's pieces: w, w + workers, ...
void work(Job &j, int w)
{
    hipError_t e = hipSetDevice(j.device);
    hipEvent_t ev[2] = {nullptr, nullptr};
    for (int k = 0; k < 2 && e == hipSuccess; ++k)
        e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
    const size_t n = (j.bytes + SLOT - 1) / SLOT;
    unsigned char *slot[2] = {j.base + (size_t)(2 * w) * SLOT, j.base + (size_t)(2 * w + 1) * SLOT};
    auto piece = [&](size_t i) { return std::min(SLOT, j.bytes - i * SLOT); };
    auto send = [&](size_t i, int k) {
        if (e != hipSuccess) return;
        if (j.up)
            e = hipMemcpyAsync(j.dev + i * SLOT, slot[k], piece(i), hipMemcpyHostToDevice, j.s);
        else
            e = hipMemcpyAsync(slot[k], j.dev + i * SLOT, piece(i), hipMemcpyDeviceToHost, j.s);
        if (e == hipSuccess) e = hipEventRecord(ev[k], j.s);
    };
    int k = 0;
    if (j.up) {
        bool used[2] = {false, false};
        for (size_t i = (size_t)w; i < n && e == hipSuccess; i += (size_t)j.workers, k ^= 1) {
            if (used[k]) e = hipEventSynchronize(ev[k]);
            if (e != hipSuccess) break;
            memcpy(slot[k], j.host + i * SLOT, piece(i));
            send(i, k);
            used[k] = true;
        }
        for (int q = 0; q < 2; ++q)
            if (used[q]) {
                const hipError_t f = hipEventSynchronize(ev[q]);
                if (e == hipSuccess) e = f;
            }
    } else {
        const size_t st = (size_t)j.workers;
        if ((size_t)w < n) send((size_t)w, 0);
        for (size_t i = (size_t)w; i < n && e == hipSuccess; i += st, k ^= 1) {
            if (i + st < n) send(i + st, k ^ 1);
            if (e == hipSuccess) e = hipEventSynchronize(ev[k]);
            if (e == hipSuccess) memcpy(j.host + i * SLOT, slot[k], piece(i));
        }
    }
    for (int q = 0; q < 2; ++q)
        if (ev[q]) (void)hipEventDestroy(ev[q]);
    if (e != hipSuccess) j.err.store((int)e);
}

hipError_t plain(void *host, void *dev, size_t bytes, bool up, hipStream_t s)
{
    if (bytes == 0) return hipSuccess;
    if (up) return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
    // up to 16 KB an asynchronous copy and a wait take 22 us, the copies that
    // wait 13 (statuses, counts, volumes and density of 500 cells 78 us, with
    // hipMemcpyWithStream 69, so 52); above they take the same
    if (bytes <= 16384) {
        const hipError_t e = hipStreamSynchronize(s);
        return e == hipSuccess ? hipMemcpy(host, dev, bytes, hipMemcpyDeviceToHost) : e;
    }
    return hipMemcpyWithStream(host, dev, bytes, hipMemcpyDeviceToHost, s);
}

// memory that the device does not reach by itself (pinned, managed and device
// memory take one plain copy)
bool pageable(const void *p)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return true;
}

hipError_t copy(void *host, void *dev, size_t bytes, bool up, hipStream_t s)
{
    if (bytes < (up ? LEAST_UP : LEAST_DOWN) || !pageable(host))
        return plain(host, dev, bytes, up, s);
    Slots &q = slots();
    std::unique_lock<std::mutex> lk(q.mu, std::try_to_lock);
    if (!lk.owns_lock()) return plain(host, dev, bytes, up, s);
    if (!q.base && hipHostMalloc((void **)&q.base, 2 * WORKERS * SLOT, hipHostMallocPortable) !=
                       hipSuccess) {
        (void)hipGetLastError();
        q.base = nullptr;
        return plain(host, dev, bytes, up, s);
    }
    Job j;
    j.host = static_cast<unsigned char *>(host);
    j.dev = static_cast<unsigned char *>(dev);
    j.bytes = bytes;
    j.up = up;
    j.s = s;
    j.base = q.base;
    hipError_t e = hipGetDevice(&j.device);
    if (e != hipSuccess) return e;
    j.workers = (int)std::min<size_t>(WORKERS, 1 + bytes / PER_WORKER);
    std::thread th[WORKERS];
    int started = 1;
    try {
        for (; started < j.workers; ++started)
            th[started] = std::thread([&j, started] { work(j, started); });
    } catch (const std::exception &) {   // no thread or memory: their pieces follow below
    }
    work(j, 0);
    for (int w = 1; w < started; ++w) th[w].join();
    for (int w = started; w < j.workers; ++w) work(j, w);
    e = (hipError_t)j.err.load();
    if (e != hipSuccess) (void)hipStreamSynchronize(s);   // no copy may still use a slot
    return e;
}

}  // namespace

void transfer_open()
{
    std::lock_guard<std::mutex> lk(slots().mu);
    ++slots().users;
}

void transfer_close()
{
    std::lock_guard<std::mutex> lk(slots().mu);
    if (--slots().users == 0 && slots().base) {
        (void)hipHostFree(slots().base);
        slots().base = nullptr;
    }
}

hipError_t copy_to_host(void *dst, const void *src, size_t bytes, hipStream_t s)
{
    return copy(dst, const_cast<void *>(src), bytes, false, s);
}

hipError_t copy_to_device(void *dst, const void *src, size_t bytes, hipStream_t s)
{
    return copy(const_cast<void *>(src), dst, bytes, true, s);
}

}  // namespace t2
