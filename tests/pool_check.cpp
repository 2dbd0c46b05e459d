// The library's block pool over a stand-in HIP runtime in host memory: one check per
// name given on the command line, exit status 0 when it holds.
#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <random>
#include <string>
#include <thread>
#include <unordered_map>
#include <utility>
#include <vector>

typedef int hipError_t;
typedef void* hipStream_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidDevice = 101 };
enum { hipStreamNonBlocking = 1 };
struct hipDeviceProp_t {
    size_t totalGlobalMem, sharedMemPerBlock;
    int multiProcessorCount;
};

// Blocks are untouched host memory until a check writes to them.
static const size_t kMiB = (size_t)1 << 20, kGiB = (size_t)1 << 30, kTotal = 12 * kGiB;
static std::mutex g_mu;
static std::unordered_map<void*, size_t> g_sizes;
static size_t g_used = 0;
static std::atomic<int> g_foreign{0};  // frees of what the runtime does not hold

static hipError_t hipMalloc(void** p, size_t n)
{
    std::lock_guard<std::mutex> lock(g_mu);
    *p = nullptr;
    if (n > kTotal || g_used + n > kTotal) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    g_sizes[*p] = n;
    g_used += n;
    return hipSuccess;
}
static hipError_t hipFree(void* p)
{
    std::lock_guard<std::mutex> lock(g_mu);
    auto it = g_sizes.find(p);
    if (it == g_sizes.end()) {
        ++g_foreign;
        return hipErrorInvalidValue;
    }
    g_used -= it->second;
    g_sizes.erase(it);
    std::free(p);
    return hipSuccess;
}
static size_t used()
{
    std::lock_guard<std::mutex> lock(g_mu);
    return g_used;
}
[[maybe_unused]] static hipError_t hipMemGetInfo(size_t* f, size_t* t)
{
    *t = kTotal;
    *f = kTotal - used();
    return hipSuccess;
}
static hipError_t hipDeviceSynchronize() { return hipSuccess; }
static hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
static hipError_t hipSetDevice(int) { return hipSuccess; }
static hipError_t hipGetLastError() { return hipSuccess; }
static const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
static hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int)
{
    *p = {kTotal, 1, 256};
    return hipSuccess;
}
static hipError_t hipStreamCreateWithFlags(hipStream_t* s, int) { *s = std::malloc(1); return hipSuccess; }
static hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
static hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }

enum { HD_OK = 0, HD_ERR_HIP = 2, HD_ERR_NOMEM = 3 };
namespace hd {
static int fail(int code, const std::string&) { return code; }
}  // namespace hd
#define HD_HIP(x)                                                  \
    do {                                                           \
        if ((x) != hipSuccess) return fail(HD_ERR_HIP, "hip call"); \
    } while (0)
#include "hd_pool.hpp"

using namespace hd;

static void* get(size_t n)
{
    void* p = nullptr;
    return dalloc(&p, n, "check") == HD_OK ? p : nullptr;
}

// Blocks of eight threads, 1 byte to 3 MB, each with its owner's mark at both ends.
static bool threads()
{
    std::atomic<int> bad{0};
    std::vector<std::thread> ts;
    for (int t = 0; t < 8; ++t)
        ts.emplace_back([&bad, t] {
            std::mt19937 g(t);
            std::vector<std::pair<unsigned char*, size_t>> held;
            const unsigned char mark = (unsigned char)(t + 1);
            for (int i = 0; i < 5000; ++i) {
                const size_t n = 1 + g() % (g() % 4 ? 4000 : 3000000);
                unsigned char* p = static_cast<unsigned char*>(get(n));
                if (!p) {
                    ++bad;
                    continue;
                }
                p[0] = p[n - 1] = mark;
                held.push_back({p, n});
                while (held.size() > 3 || (i == 4999 && !held.empty())) {
                    const size_t k = g() % held.size();
                    const auto h = held[k];
                    held.erase(held.begin() + (long)k);
                    if (h.first[0] != mark || h.first[h.second - 1] != mark) ++bad;
                    if (dfree_status(h.first) != hipSuccess) ++bad;
                }
                if (i % 50 == 0) {
                    hipStream_t s = nullptr;
                    if (stream_get(&s) != hipSuccess) ++bad;
                    stream_put(s);
                }
            }
        });
    for (auto& t : ts) t.join();
    const auto& d = pool().dev[0];
    return !bad && !g_foreign && d.live_bytes == 0 && d.idle_bytes == used();
}

static bool twice()
{
    void *keep = get(16), *p = get(100);
    bool ok = dfree_status(p) == hipSuccess && dfree_status(p) == hipErrorInvalidValue;
    void *a = get(100), *b = get(100);
    ok = ok && a && b && a != b;
    dfree(a);
    dfree(b);
    dfree(keep);
    return ok && !g_foreign && pool().dev[0].idle_bytes == used();
}

static bool sizes()
{
    for (size_t n : {(size_t)0, (size_t)1, (size_t)256, (size_t)257, kMiB, kMiB + 1, 2 * kMiB - 1, 2 * kMiB, 2 * kMiB + 1}) {
        void* p = get(n);
        if (!p) return false;
        {
            std::lock_guard<std::mutex> lock(g_mu);
            if (g_sizes[p] < n) return false;
        }
        dfree(p);
    }
    for (size_t n : {SIZE_MAX, SIZE_MAX - kMiB, SIZE_MAX - 2 * kMiB + 2, SIZE_MAX / 2, kTotal + 1})
        if (get(n)) return false;
    return true;
}

// A request that fits only without the idle blocks.
static bool drain()
{
    void *keep = get(16), *a = get(kGiB / 2), *b = get(kGiB / 2);
    dfree(a);
    dfree(b);
    const bool idle = used() >= kGiB;
    void* p = get(kTotal - kGiB / 4);
    const bool ok = idle && p;
    dfree(p);
    dfree(keep);
    return ok;
}

static bool bounded()
{
    void* keep = get(16);
    std::vector<void*> v;
    for (int i = 0; i < 6; ++i) v.push_back(get(kGiB));
    for (void* p : v) dfree(p);
    const bool ok = used() <= kTotal / 6 + kMiB;
    dfree(keep);
    return ok && used() <= 256 * kMiB;  // nothing is in use
}

// Most of the device in use: what is returned leaves three quarters of the rest.
static bool quarter()
{
    void *keep = get(16), *big = get(5 * kGiB);
    std::vector<void*> v;
    for (int i = 0; i < 6; ++i) v.push_back(get(kGiB));
    const size_t rest = kTotal - used() + 6 * kGiB;
    for (void* p : v) dfree(p);
    const bool ok = kTotal - used() >= rest * 3 / 4 && used() >= 6 * kGiB;  // some of it is kept
    dfree(big);
    dfree(keep);
    return ok;
}

static bool trim()
{
    void* keep = get(16);
    std::vector<void*> v;
    for (int i = 0; i < 4; ++i) v.push_back(get(kGiB / 4));
    for (void* p : v) dfree(p);
    size_t idle = 0;
    bool ok = used() >= kGiB && pool_trim(kGiB / 2, &idle) == HD_OK && idle <= kGiB / 2 && idle >= kGiB / 4;
    ok = ok && pool_trim(0, &idle) == HD_OK && idle == 0 && used() < kMiB;
    dfree(keep);
    return ok && pool_trim(0, nullptr) == HD_OK && used() == 0;
}

int main(int argc, char** argv)
{
    const std::pair<const char*, bool (*)()> checks[] = {
        {"threads", threads}, {"twice", twice}, {"sizes", sizes}, {"drain", drain}, {"bounded", bounded},
        {"quarter", quarter}, {"trim", trim}};
    for (const auto& c : checks)
        if (argc == 2 && !std::strcmp(argv[1], c.first)) return c.second() ? 0 : 1;
    return 2;
}
