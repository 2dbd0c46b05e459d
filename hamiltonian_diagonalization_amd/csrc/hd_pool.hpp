// The library's device blocks and streams, included by hd_basis.hip.  It calls the HIP
// runtime only through hipMalloc, hipFree, hipMemGetInfo, the device and the stream
// calls, so the bookkeeping also compiles against a stand-in runtime on the CPU.
#pragma once

#include <algorithm>
#include <chrono>
#include <cstdint>
#include <iterator>
#include <map>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

namespace hd {

// ------------------------------------------------- device memory and streams
//
// Blocks and streams are kept for reuse: a build, a solve or a sweep point asks
// for the sizes that the previous one returned, and mapping and clearing gigabytes
// anew cost more than the kernels that fill them.
// Builds in a loop, the previous result still held: N=10, 2S=27 in every format
// 7-22 -> 2.3 ms, the 6x5 N=6 Wannier sector 105-190 -> 39 ms, N=12, 2S=33 coded
// build + tiled layout + product 190-770 -> 190 ms.  A stream costs about 0.5 ms
// to create and destroy (57 builds of a batch: 348 -> 317 ms with the solve).
//
// Bounds: idle blocks of a device never exceed a sixth of its memory, nor, above
// kUnasked, a quarter of what would be free without them when a block is returned, so
// that other allocators of the process and other processes find three quarters of it.
// The driver's answer takes 10 us (asked at each return, a build of 0.9 GB was 3% and a
// basis of 8,512 states 30% slower), so it stands for kAskAgain.  They go back to the
// driver down to kKeepBytes when the device's last live block is returned, entirely
// when an allocation of the library fails, and on request (hd_mem_trim).  A returned
// block is idle only after the whole device has finished its work (hipFree waits in
// the same way), so it may be handed to any thread and any stream.  The pool is never
// destroyed: handles may be released while the process ends.
namespace {
constexpr int kPoolDevices = 64;
constexpr size_t kKeepBytes = (size_t)256 << 20;
constexpr size_t kUnasked = (size_t)1 << 30;
constexpr std::chrono::milliseconds kAskAgain(10);
constexpr size_t kKeepStreams = 64;  // idle streams per device

struct PoolDevice {
    std::multimap<size_t, void*> idle;  // by size
    size_t idle_bytes = 0, live_bytes = 0, cap = 0;
    size_t bound = 0;  // of idle_bytes, as of `asked`
    std::chrono::steady_clock::time_point asked;
    std::vector<hipStream_t> streams;
    int n_cu = 0;
    size_t max_lds = 0;
};

struct Pool {
    struct Block {
        size_t bytes;
        int dev;
        bool live;  // handed out; false while it is returned and idle
    };
    std::mutex mu;
    std::unordered_map<void*, Block> blocks;  // every block that the driver has given and not got back
    std::unordered_map<hipStream_t, int> stream_dev;
    PoolDevice dev[kPoolDevices];
};

Pool& pool()
{
    static Pool* p = new Pool;
    return *p;
}

// Powers of two up to 1 MiB, then multiples of 2 MiB; 0 where that exceeds size_t.
size_t pool_size(size_t bytes)
{
    constexpr size_t step = (size_t)2 << 20;
    if (bytes > SIZE_MAX - (step - 1)) return 0;
    if (bytes > (size_t)1 << 20) return (bytes + step - 1) / step * step;
    size_t s = 256;
    while (s < bytes) s <<= 1;
    return s;
}

// Takes idle blocks of `d` (largest first) until at most `keep` bytes stay.
void pool_take_excess(Pool& P, PoolDevice& d, size_t keep, std::vector<void*>& out)
{
    while (d.idle_bytes > keep && !d.idle.empty()) {
        auto it = std::prev(d.idle.end());
        d.idle_bytes -= it->first;
        out.push_back(it->second);
        P.blocks.erase(it->second);
        d.idle.erase(it);
    }
}

// Runs f with `dev` current.
template <typename F>
void on_device(int dev, F f)
{
    int cur = dev;
    (void)hipGetDevice(&cur);
    if (cur != dev) (void)hipSetDevice(dev);
    f();
    if (cur != dev) (void)hipSetDevice(cur);
}

// The device's constants, read once.
hipError_t pool_device(int dev)
{
    Pool& P = pool();
    {
        std::lock_guard<std::mutex> lock(P.mu);
        if (P.dev[dev].n_cu) return hipSuccess;
    }
    hipDeviceProp_t prop;
    const hipError_t e = hipGetDeviceProperties(&prop, dev);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lock(P.mu);
    P.dev[dev].cap = prop.totalGlobalMem / 6;
    P.dev[dev].max_lds = prop.sharedMemPerBlock;
    P.dev[dev].n_cu = prop.multiProcessorCount;
    return hipSuccess;
}
}  // namespace

int dalloc(void** p, size_t bytes, const char* what)
{
    *p = nullptr;
    Pool& P = pool();
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess && (dev < 0 || dev >= kPoolDevices)) e = hipErrorInvalidDevice;
    if (e == hipSuccess) e = pool_device(dev);
    const size_t need = pool_size(bytes);
    if (e == hipSuccess && !need) e = hipErrorOutOfMemory;
    if (e == hipSuccess) {
        {
            std::lock_guard<std::mutex> lock(P.mu);
            PoolDevice& d = P.dev[dev];
            auto it = d.idle.lower_bound(need);
            if (it != d.idle.end() && it->first <= need + need / 8) {
                *p = it->second;
                P.blocks[*p].live = true;
                d.live_bytes += it->first;
                d.idle_bytes -= it->first;
                d.idle.erase(it);
                return HD_OK;
            }
        }
        size_t got = need;
        e = hipMalloc(p, got);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            std::vector<void*> drop;
            {
                std::lock_guard<std::mutex> lock(P.mu);
                pool_take_excess(P, P.dev[dev], 0, drop);
            }
            for (void* q : drop) (void)hipFree(q);
            got = std::max<size_t>(bytes, 16);  // without the rounding: what was asked for may still fit
            e = hipMalloc(p, got);
        }
        if (e == hipSuccess) {
            std::lock_guard<std::mutex> lock(P.mu);
            P.blocks[*p] = {got, dev, true};
            P.dev[dev].live_bytes += got;
            return HD_OK;
        }
    }
    (void)hipGetLastError();
    *p = nullptr;
    return fail(HD_ERR_NOMEM, std::string("hipMalloc of ") + std::to_string(bytes) +
                                  " bytes for " + what + " failed: " + hipGetErrorString(e));
}

hipError_t dfree_status(void* p)
{
    if (!p) return hipSuccess;
    Pool& P = pool();
    Pool::Block b;
    {
        std::lock_guard<std::mutex> lock(P.mu);
        auto it = P.blocks.find(p);
        if (it == P.blocks.end()) return hipFree(p);  // not from dalloc: the driver's answer
        // Given back already.  The driver still has the block as allocated and would
        // free it under the idle list.
        if (!it->second.live) return hipErrorInvalidValue;
        it->second.live = false;
        b = it->second;
        P.dev[b.dev].live_bytes -= b.bytes;
    }
    hipError_t e = hipSuccess;
    std::vector<void*> drop;
    on_device(b.dev, [&]() {
        e = hipDeviceSynchronize();
        {
            std::lock_guard<std::mutex> lock(P.mu);
            PoolDevice& d = P.dev[b.dev];
            const size_t all = d.idle_bytes + b.bytes;
            size_t bound = d.live_bytes ? std::min(d.cap, kUnasked) : kKeepBytes;
            if (d.live_bytes && all > bound) {
                const auto now = std::chrono::steady_clock::now();
                if (all > d.bound || now - d.asked > kAskAgain) {
                    size_t free_ = 0, total = 0;
                    if (hipMemGetInfo(&free_, &total) != hipSuccess) free_ = 0;
                    d.bound = std::min(d.cap, std::max(kUnasked, (free_ + all) / 4));
                    d.asked = now;
                }
                bound = d.bound;
            }
            if (e == hipSuccess && all <= bound) {
                d.idle.emplace(b.bytes, p);
                d.idle_bytes += b.bytes;
            } else {
                P.blocks.erase(p);
                drop.push_back(p);
            }
            pool_take_excess(P, d, bound, drop);
        }
        for (void* q : drop) {
            const hipError_t f = hipFree(q);
            if (e == hipSuccess) e = f;
        }
    });
    return e;
}

void dfree(void* p) { (void)dfree_status(p); }

// hd_mem_trim
int pool_trim(size_t keep, size_t* idle)
{
    int dev = -1;
    HD_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kPoolDevices) return fail(HD_ERR_HIP, "device index beyond the pool's table");
    Pool& P = pool();
    std::vector<void*> drop;
    {
        std::lock_guard<std::mutex> lock(P.mu);
        pool_take_excess(P, P.dev[dev], keep, drop);
        if (idle) *idle = P.dev[dev].idle_bytes;
    }
    hipError_t e = hipSuccess;
    for (void* q : drop) {
        const hipError_t f = hipFree(q);
        if (e == hipSuccess) e = f;
    }
    HD_HIP(e);
    return HD_OK;
}

hipError_t stream_get(hipStream_t* s)
{
    *s = nullptr;
    Pool& P = pool();
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kPoolDevices) return hipErrorInvalidDevice;
    {
        std::lock_guard<std::mutex> lock(P.mu);
        auto& v = P.dev[dev].streams;
        if (!v.empty()) {
            *s = v.back();
            v.pop_back();
            P.stream_dev[*s] = dev;
            return hipSuccess;
        }
    }
    e = hipStreamCreateWithFlags(s, hipStreamNonBlocking);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lock(P.mu);
    P.stream_dev[*s] = dev;
    return hipSuccess;
}

void stream_put(hipStream_t s)
{
    if (!s) return;
    Pool& P = pool();
    const bool idle = hipStreamSynchronize(s) == hipSuccess;
    {
        std::lock_guard<std::mutex> lock(P.mu);
        auto it = P.stream_dev.find(s);
        if (it != P.stream_dev.end()) {
            auto& v = P.dev[it->second].streams;
            P.stream_dev.erase(it);
            if (idle && v.size() < kKeepStreams) {
                v.push_back(s);
                return;
            }
        }
    }
    (void)hipStreamDestroy(s);
}

}  // namespace hd
