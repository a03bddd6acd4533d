// tsp_mem.hip -- device memory behind tsp_malloc / tsp_free and the device
// conversions.
//
// hipMalloc and hipFree cost 40-230 us each on MI355X, and the driver clears
// recycled VRAM at about 30 GB/s before it hands it out again: a program that
// converts one matrix after another spent 145 of 179 ms (RMAT scale 22, 4.6
// GB of tiles) and 0.6 of 0.94 ms (a circuit of 117k rows) in them.  Freed
// blocks are therefore kept for the next request of about their size:
//   * a block is one whole hipMalloc allocation, never a part of one, so a
//     caller may also hand it to hipFree;
//   * a block comes back only after its device is idle (as with hipFree), or
//     when the caller has waited for the only stream that used it;
//   * idle blocks hold at most 1/32 of the device's memory (9 GB); the least
//     recently used go first, and any that kIdleCalls requests have passed
//     over.  tsp_mem_trim, and a hipMalloc that fails, give all back;
//   * a block's range is checked with the runtime before it is kept or
//     reused, so one that was freed behind this file's back (hipFree,
//     hipDeviceReset) is forgotten.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <list>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "../../include/tilespmm_hip.h"
#include "tsp_kernels.h"

namespace {

constexpr unsigned long long kIdleCalls = 256;

struct Block {
    void *p;
    size_t bytes;        // asked of hipMalloc
    size_t range;        // what the runtime reports for it
    int dev;
    unsigned long long used;
};

struct Pool {
    std::mutex mu;
    std::unordered_map<void *, Block> out;      // handed out
    std::list<Block> idle;                      // least recently used first
    unsigned long long clock = 0;
};

// never destroyed: the HIP runtime may be gone when static objects are
Pool &pool()
{
    static Pool *p = new Pool;
    return *p;
}

// Sizes in steps of 1/16 of their power of two, so that requests that differ
// a little share blocks.
size_t step_up(size_t n)
{
    size_t s = 4096;
    while (s * 32 <= n) s *= 2;
    return (n + s - 1) / s * s;
}

bool still_ours(const Block &b)
{
    hipDeviceptr_t base = nullptr;
    size_t range = 0;
    if (hipMemGetAddressRange(&base, &range, (hipDeviceptr_t)b.p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return (void *)base == b.p && range == b.range;
}

size_t idle_limit(int dev)
{
    size_t total = 0;
    if (hipDeviceTotalMem(&total, dev) != hipSuccess) return 0;
    return total / 32;
}

void give_back(const std::vector<Block> &gone)
{
    for (const Block &b : gone) {
        if (!still_ours(b)) continue;
        (void)hipFree(b.p);
    }
    if (!gone.empty()) (void)hipGetLastError();
}

void trim_device(int dev)            // dev < 0: every device
{
    std::vector<Block> gone;
    {
        Pool &pl = pool();
        std::lock_guard<std::mutex> lock(pl.mu);
        for (auto it = pl.idle.begin(); it != pl.idle.end();)
            if (dev < 0 || it->dev == dev) {
                gone.push_back(*it);
                it = pl.idle.erase(it);
            } else {
                ++it;
            }
    }
    give_back(gone);
}

}  // namespace

namespace tsp {

int dev_alloc(void **ptr, size_t bytes)
{
    *ptr = nullptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    const size_t want = step_up(bytes ? bytes : 16);
    Pool &pl = pool();
    for (;;) {
        Block got{};
        {
            std::lock_guard<std::mutex> lock(pl.mu);
            ++pl.clock;
            auto best = pl.idle.end();
            for (auto it = pl.idle.begin(); it != pl.idle.end(); ++it)
                if (it->dev == dev && it->bytes >= want && it->bytes - want <= want / 4 &&
                    (best == pl.idle.end() || it->bytes < best->bytes))
                    best = it;
            if (best == pl.idle.end()) break;
            got = *best;
            pl.idle.erase(best);
        }
        if (!still_ours(got)) continue;
        std::lock_guard<std::mutex> lock(pl.mu);
        pl.out[got.p] = got;
        *ptr = got.p;
        return TSP_OK;
    }
    void *p = nullptr;
    e = hipMalloc(&p, want);
    if (e != hipSuccess) {
        (void)hipGetLastError();      // must not surface as the error of a later launch
        trim_device(dev);
        e = hipMalloc(&p, bytes ? bytes : 16);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            return (int)e;
        }
    }
    Block b{p, want, 0, dev, 0};
    hipDeviceptr_t base = nullptr;
    if (hipMemGetAddressRange(&base, &b.range, (hipDeviceptr_t)p) == hipSuccess && (void *)base == p && b.range >= want) {
        std::lock_guard<std::mutex> lock(pl.mu);
        pl.out[p] = b;                // (replaces an entry that hipFree made stale)
    } else {
        (void)hipGetLastError();      // not kept: tsp_free hands it to hipFree
        std::lock_guard<std::mutex> lock(pl.mu);
        pl.out.erase(p);
    }
    *ptr = p;
    return TSP_OK;
}

int dev_free(void *ptr, bool waited)
{
    if (!ptr) return TSP_OK;
    Pool &pl = pool();
    Block b{};
    {
        std::lock_guard<std::mutex> lock(pl.mu);
        auto it = pl.out.find(ptr);
        if (it != pl.out.end()) {
            b = it->second;
            pl.out.erase(it);
        }
    }
    const size_t limit = b.p ? idle_limit(b.dev) : 0;
    if (!b.p || b.bytes > limit || !still_ours(b)) return (int)hipFree(ptr);
    if (!waited) {
        // work on any stream may still use the block
        int cur = 0;
        hipError_t e = hipGetDevice(&cur);
        if (e == hipSuccess && cur != b.dev) e = hipSetDevice(b.dev);
        if (e == hipSuccess) e = hipDeviceSynchronize();
        if (cur != b.dev) (void)hipSetDevice(cur);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            return (int)hipFree(ptr);
        }
    }
    std::vector<Block> gone;
    {
        std::lock_guard<std::mutex> lock(pl.mu);
        b.used = ++pl.clock;
        pl.idle.push_back(b);
        size_t sum = 0;
        for (const Block &x : pl.idle) sum += x.dev == b.dev ? x.bytes : 0;
        for (auto it = pl.idle.begin(); it != pl.idle.end();) {
            const bool over = it->dev == b.dev && sum > limit, old = pl.clock - it->used > kIdleCalls;
            if (over) sum -= it->bytes;
            if (over || old) {
                gone.push_back(*it);
                it = pl.idle.erase(it);
            } else {
                ++it;
            }
        }
    }
    give_back(gone);
    return TSP_OK;
}

}  // namespace tsp

extern "C" {

int tsp_malloc(void **ptr, size_t bytes)
{
    if (!ptr) return TSP_EINVAL;
    *ptr = nullptr;
    return bytes == 0 ? TSP_OK : tsp::dev_alloc(ptr, bytes);
}

int tsp_free(void *ptr) { return tsp::dev_free(ptr, false); }

int tsp_mem_trim(void)
{
    trim_device(-1);
    return TSP_OK;
}

}  // extern "C"
