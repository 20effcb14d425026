// Large copies between device memory and a caller's pageable host memory.
//
// hipMemcpyAsync on pageable memory copies through the runtime's staging buffer with one host thread, which
// also takes the page faults of fresh destination pages: 7-10 GB/s out of and 28 GB/s into the device.
// Here the chunks of a copy pass through a ring of pinned slots: the calling thread alone talks to the
// runtime, keeping the ring's DMA transfers queued on the caller's stream, and STAGE_WORKERS
// threads copy between the slots and the host memory, faults and all, beside each other and the
// transfers.  (Threads that each issued and awaited their own chunks' transfers lost 100 us a chunk to
// each other in the runtime.)
//
// The slots belong to the device and not to a handle (STAGE_SLOTS x STAGE_CHUNK), made at the first large copy
// and given back with the device's last handle.  One copy uses them at a time; a copy that finds them taken
// (another thread's handle), that is small, or whose host memory is not pageable goes through
// hipMemcpyAsync.
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

#include "axg_internal.h"

namespace axg {

namespace {

constexpr int STAGE_WORKERS = 7, STAGE_SLOTS = 8;
constexpr size_t STAGE_CHUNK = (size_t)4 << 20;
// Two fields out / in, ms, hipMemcpyAsync -> this: 128^3 (32 MiB each) 6.7 / 2.2 -> 4.5 / 2.0, 256^3 51 / 17.5 ->
// 29 / 12 (13 / 12 with a warmed DMA engine), 512^3 410 / 139 -> 95 / 93 (46 GB/s each way); a 512^3
// flag plane 13 -> 3.4.  Chunks of 2 MiB 109 / 107 and of 1 MiB 143 / 144 at 512^3; 4 workers 103, 11 workers
// 94.  Below 16 MiB the gain (96^3 3.3 -> 2.5 out, 0.85 -> 1.0 in) does not pay the ring's making, 3 ms once.
constexpr size_t STAGE_MIN = (size_t)16 << 20;
constexpr int STAGE_DEVICES = 16;

struct Pool {
    std::mutex busy;   // held by the copy that uses the chunks
    std::mutex users;  // guards n
    int n = 0;         // handles on the device
    void* buf[STAGE_SLOTS] = {};
    hipEvent_t ev[STAGE_SLOTS] = {};

    bool ready()
    {
        for (int t = 0; t < STAGE_SLOTS; t++) {
            if (!buf[t] && hipHostMalloc(&buf[t], STAGE_CHUNK, hipHostMallocDefault) != hipSuccess) buf[t] = nullptr;
            if (!ev[t] && hipEventCreateWithFlags(&ev[t], hipEventDisableTiming) != hipSuccess) ev[t] = nullptr;
            if (!buf[t] || !ev[t]) {
                (void)hipGetLastError();
                return false;
            }
        }
        return true;
    }
    void give_back()
    {
        for (int t = 0; t < STAGE_SLOTS; t++) {
            if (buf[t]) (void)hipHostFree(buf[t]);
            if (ev[t]) (void)hipEventDestroy(ev[t]);
            buf[t] = nullptr;
            ev[t] = nullptr;
        }
    }
};

Pool g_pool[STAGE_DEVICES];

bool pageable(const void* p)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

// `bytes` through the pool's slots; false: not done this way.
bool staged(int device, hipStream_t s, char* dst, const char* src, size_t bytes, bool to_host)
{
    if (bytes < STAGE_MIN || device < 0 || device >= STAGE_DEVICES || !pageable(to_host ? dst : src)) return false;
    Pool& p = g_pool[device];
    std::unique_lock<std::mutex> lock(p.busy, std::try_to_lock);
    if (!lock.owns_lock() || !p.ready()) return false;
    const int64_t nc = (int64_t)((bytes + STAGE_CHUNK - 1) / STAGE_CHUNK);
    auto len = [&](int64_t c) { return std::min(STAGE_CHUNK, bytes - (size_t)c * STAGE_CHUNK); };
    // chunk c passes through slot c % STAGE_SLOTS.  dma: chunks transferred (in order); host[slot]: one past the
    // last chunk whose host copy through the slot is done.  All under m.  Who waits sleeps, on moved for dma and on
    // copied for host: spinning took 0.73 s of processors for two fields in at 512^3 instead of 0.27 (out
    // 0.75 and 0.44) and was no faster, at 108^3 neither (1.26 ms out, two fields, both ways).
    std::mutex m;
    std::condition_variable moved, copied;
    int64_t dma = 0, host[STAGE_SLOTS] = {};
    bool stop = false;
    std::atomic<int64_t> next{0};
    auto worker = [&] {
        for (;;) {
            const int64_t c = next.fetch_add(1);
            if (c >= nc) return;
            const int sl = (int)(c % STAGE_SLOTS);
            // out: the chunk has arrived; in: the slot's last chunk has left
            {
                std::unique_lock<std::mutex> l(m);
                moved.wait(l, [&] { return stop || dma > (to_host ? c : c - STAGE_SLOTS); });
                if (stop) return;
            }
            char* h = (to_host ? dst : const_cast<char*>(src)) + (size_t)c * STAGE_CHUNK;
            if (to_host) memcpy(h, p.buf[sl], len(c));
            else memcpy(p.buf[sl], h, len(c));
            {
                std::lock_guard<std::mutex> l(m);
                host[sl] = c + 1;
            }
            copied.notify_one();
        }
    };
    std::vector<std::thread> pool;
    try {
        const int nt = (int)std::min<int64_t>({(int64_t)STAGE_WORKERS, nc, (int64_t)std::max(1u, std::thread::hardware_concurrency())});
        pool.reserve(nt);
        for (int t = 0; t < nt; t++) pool.emplace_back(worker);
    } catch (...) {
        if (pool.empty()) return false;  // no thread to be had
    }
    hipError_t e = hipSuccess;
    int64_t queued = 0, arrived = 0;
    while (arrived < nc && e == hipSuccess) {
        // queue transfers as far as the ring and the host copies allow, wait for the oldest
        while (queued < nc && queued < arrived + STAGE_SLOTS && e == hipSuccess) {
            const int sl = (int)(queued % STAGE_SLOTS);
            const int64_t need = to_host ? queued - STAGE_SLOTS + 1 : queued + 1;
            {
                std::unique_lock<std::mutex> l(m);
                if (host[sl] < need) {
                    if (queued > arrived) break;
                    copied.wait(l, [&] { return host[sl] >= need; });
                }
            }
            const size_t at = (size_t)queued * STAGE_CHUNK;
            e = to_host ? hipMemcpyAsync(p.buf[sl], src + at, len(queued), hipMemcpyDeviceToHost, s)
                        : hipMemcpyAsync(dst + at, p.buf[sl], len(queued), hipMemcpyHostToDevice, s);
            if (e == hipSuccess) e = hipEventRecord(p.ev[sl], s);
            queued++;
        }
        if (e == hipSuccess) e = hipEventSynchronize(p.ev[arrived % STAGE_SLOTS]);
        if (e == hipSuccess) {
            {
                std::lock_guard<std::mutex> l(m);
                dma = ++arrived;
            }
            moved.notify_all();
        }
    }
    if (e != hipSuccess) {
        {
            std::lock_guard<std::mutex> l(m);
            stop = true;
        }
        moved.notify_all();
    }
    for (auto& t : pool) t.join();
    if (e != hipSuccess) {
        // nothing may still write a slot when the next copy takes it
        (void)hipStreamSynchronize(s);
        throw Error(AXG_EDEVICE, std::string("host copy: ") + hipGetErrorString(e));
    }
    return true;
}

}  // namespace

void staging_retain(int device)
{
    if (device < 0 || device >= STAGE_DEVICES) return;
    std::lock_guard<std::mutex> l(g_pool[device].users);
    g_pool[device].n++;
}

void staging_release(int device)
{
    if (device < 0 || device >= STAGE_DEVICES) return;
    Pool& p = g_pool[device];
    std::lock_guard<std::mutex> l(p.users);
    if (--p.n > 0) return;
    std::lock_guard<std::mutex> b(p.busy);
    p.give_back();
}

void copy_to_host(int device, hipStream_t s, void* dst, const void* src, size_t bytes, bool wait)
{
    if (staged(device, s, (char*)dst, (const char*)src, bytes, true)) return;
    AXG_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
    if (wait) AXG_HIP(hipStreamSynchronize(s));
}

void copy_to_device(int device, hipStream_t s, void* dst, const void* src, size_t bytes)
{
    if (staged(device, s, (char*)dst, (const char*)src, bytes, false)) return;
    AXG_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
}

}  // namespace axg
