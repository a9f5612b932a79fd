// Host-only test of the copies between host memory and the device (spcomm3d_amd/csrc/host_stage.cpp)
// where pinned memory runs out, and of the contexts' pools of device memory (dev_pool.h) where
// device memory does: over a stand-in for the few HIP calls they make, in which "device" memory is
// host memory and what can be had of either is set by the test.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <random>
#include <thread>
#include <vector>

#include "../../spcomm3d_amd/csrc/dev_pool.h"
#include "../../spcomm3d_amd/csrc/host_stage.h"

using namespace spc3d;

static int g_fail = 0;
#define CHECK(cond)                                                                               \
    do {                                                                                          \
        if (!(cond)) {                                                                            \
            std::printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond);                           \
            ++g_fail;                                                                             \
        }                                                                                         \
    } while (0)

// ---- the stand-in ------------------------------------------------------------------------
static std::mutex g_mu;
static size_t g_pinned_room;            // bytes of pinned memory that can still be had
static std::map<void *, size_t> g_pinned;
static size_t pinned_now()
{
    size_t n = 0;
    for (auto &p : g_pinned)
        n += p.second;
    return n;
}

static size_t g_device_room;
static std::map<void *, size_t> g_device;

extern "C" {
hipError_t hipMalloc(void **p, size_t n)
{
    std::lock_guard<std::mutex> lock(g_mu);
    if (n > g_device_room)
        return hipErrorOutOfMemory;
    *p = std::malloc(1);
    g_device[*p] = n;
    g_device_room -= n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> lock(g_mu);
    CHECK(g_device.count(p) == 1);
    g_device_room += g_device[p];
    g_device.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> lock(g_mu);
    *p = nullptr;
    if (n > g_pinned_room)
        return hipErrorOutOfMemory;
    *p = std::malloc(n);
    g_pinned[*p] = n;
    g_pinned_room -= n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    std::lock_guard<std::mutex> lock(g_mu);
    CHECK(g_pinned.count(p) == 1);
    g_pinned_room += g_pinned[p];
    g_pinned.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(to, from, n);
    return hipSuccess;
}
}

// ---- copies with none, some and all of the pinned memory they would use -------------------
static void copies(size_t room, unsigned threads)
{
    g_pinned_room = room;
    std::mt19937_64 g(7);
    HostStage stage;
    for (size_t bytes : {(size_t)4, (size_t)4096, (size_t)1 << 19, ((size_t)1 << 19) + 4, (size_t)9 << 20,
                         ((size_t)21 << 20) + 12}) {
        std::vector<char> src(bytes), dev(bytes, 1), back(bytes, 2);
        for (auto &c : src)
            c = (char)g();
        CHECK(stage.upload(0, dev.data(), src.data(), bytes, nullptr) == hipSuccess);
        CHECK(dev == src);
        CHECK(stage.download(0, back.data(), dev.data(), bytes, nullptr, nullptr, threads) == hipSuccess);
        CHECK(back == src);
        std::vector<BlockKey> want, keys((bytes + kKeyBlockBytes - 1) / kKeyBlockBytes);
        keys_of(src.data(), bytes, want, 1);
        std::fill(back.begin(), back.end(), 3);
        CHECK(stage.download(0, back.data(), dev.data(), bytes, nullptr, keys.data(), threads) == hipSuccess);
        CHECK(back == src);
        CHECK(keys == want);
        CHECK(pinned_now() <= room);
    }
    stage.release();
    CHECK(g_pinned.empty());
}

// A small transfer holds little pinned memory.
static void small_transfers_pin_little()
{
    g_pinned_room = (size_t)1 << 30;
    HostStage stage;
    char host[64] = {}, dev[64] = {};
    CHECK(stage.download(0, host, dev, sizeof host, nullptr, nullptr, 8) == hipSuccess);
    CHECK(stage.upload(0, dev, host, sizeof host, nullptr) == hipSuccess);
    CHECK(pinned_now() > 0 && pinned_now() <= (size_t)2 << 20);
}

// What one context's pool keeps gives way to another context that runs out; other devices' pools
// and blocks in use do not.
static void pools_give_way()
{
    g_device_room = 100 << 10;
    {
        DevPool a, b, other;
        a.open(0, 90 << 10);
        b.open(0, 90 << 10);
        other.open(1, 90 << 10);
        void *p = nullptr, *q = nullptr, *r = nullptr, *s = nullptr;
        CHECK(a.get(&p, 40 << 10) == hipSuccess && a.get(&q, 20 << 10) == hipSuccess);
        CHECK(other.get(&r, 20 << 10) == hipSuccess);
        a.put(p);
        other.put(r);
        CHECK(g_device.size() == 3);
        CHECK(b.get(&s, 50 << 10) == hipSuccess && s); // fits once a's 40 KiB are free
        CHECK(g_device.size() == 3 && g_device.count(q) && g_device.count(r));
        b.put(s);
        CHECK(DevPool::device_alloc(0, &p, 60 << 10) == hipSuccess); // a panel's: b's 50 KiB give way
        CHECK(b.get(&s, 30 << 10) == hipErrorOutOfMemory && s == nullptr);
        CHECK(hipFree(p) == hipSuccess);
        a.put(q);
    }
    CHECK(g_device.empty());
    std::vector<std::thread> threads; // pools made, run dry and dropped side by side
    g_device_room = 400 << 10;
    for (int t = 0; t < 4; ++t)
        threads.emplace_back([t] {
            std::mt19937 g(t);
            for (int round = 0; round < 200; ++round) {
                DevPool pool;
                pool.open(t % 2, 200 << 10);
                std::vector<void *> held;
                for (int i = 0; i < 12; ++i) {
                    void *p = nullptr;
                    if (pool.get(&p, (g() % 64 + 1) << 10) == hipSuccess)
                        held.push_back(p);
                    if (!held.empty() && g() % 2) {
                        pool.put(held.back());
                        held.pop_back();
                    }
                }
                for (void *p : held)
                    pool.put(p);
            }
        });
    for (auto &t : threads)
        t.join();
    CHECK(g_device.empty());
}

// A kept block serves what is smaller by up to the caller's spare, by a quarter unless it says otherwise.
static void kept_blocks_serve_smaller_ones()
{
    g_device_room = 400 << 10;
    {
        DevPool a;
        a.open(0, 400 << 10);
        void *p = nullptr, *q = nullptr;
        CHECK(a.get(&p, 100 << 10) == hipSuccess);
        a.put(p);
        CHECK(a.get(&q, 80 << 10) == hipSuccess && q == p);
        a.put(q);
        CHECK(a.get(&q, (80 << 10) - 512) == hipSuccess && q != p);
        a.put(q); // (kept: 100 KiB and half a KiB less than 80)
        CHECK(a.get(&q, 50 << 10, 50 << 10) == hipSuccess && q != p); // the smaller of two that would do
        void *r = nullptr;
        CHECK(a.get(&r, 50 << 10, (50 << 10) - 1) == hipSuccess && r != p && r != q);
        a.put(r);
        CHECK(a.get(&r, 51 << 10, 49 << 10) == hipSuccess && r == p);
        a.put(r);
        a.put(q);
    }
    CHECK(g_device.empty());
}

int main()
{
    pools_give_way();
    kept_blocks_serve_smaller_ones();
    for (unsigned threads : {1u, 3u})
        for (size_t room : {(size_t)0, (size_t)1 << 20, (size_t)2 << 20, (size_t)13 << 20, (size_t)30 << 20,
                            (size_t)1 << 30})
            copies(room, threads);
    small_transfers_pin_little();
    CHECK(g_pinned.empty());
    std::printf(g_fail ? "FAILED (%d)\n" : "PASSED\n", g_fail);
    return g_fail != 0;
}
