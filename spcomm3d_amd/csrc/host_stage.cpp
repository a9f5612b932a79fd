// Copies between pageable host memory and the device (see host_stage.h).
#include "host_stage.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <new>
#include <system_error>
#include <thread>

namespace spc3d {

hipError_t HostStage::lane(unsigned i, Lane **out)
{
    *out = nullptr;
    try {
        while (lanes_.size() <= i) {
            std::unique_ptr<Lane> l(new Lane());
            hipError_t e = hipHostMalloc((void **)&l->buf, kMaxPiece * kBufs, hipHostMallocDefault);
            for (unsigned b = 0; b < kBufs && e == hipSuccess; ++b)
                e = hipEventCreateWithFlags(&l->ev[b], hipEventDisableTiming);
            if (e != hipSuccess) {
                for (hipEvent_t ev : l->ev)
                    if (ev) (void)hipEventDestroy(ev);
                if (l->buf) (void)hipHostFree(l->buf);
                return e;
            }
            lanes_.push_back(std::move(l));
        }
    } catch (const std::bad_alloc &) {
        return hipErrorOutOfMemory;
    }
    *out = lanes_[i].get();
    return hipSuccess;
}

void HostStage::release()
{
    std::lock_guard<std::mutex> lock(mu_);
    for (auto &l : lanes_) {
        for (unsigned b = 0; b < kBufs; ++b) {
            (void)wait(*l, b);
            (void)hipEventDestroy(l->ev[b]);
        }
        (void)hipHostFree(l->buf);
    }
    lanes_.clear();
}

hipError_t HostStage::wait(Lane &l, unsigned b)
{
    if (!l.busy[b])
        return hipSuccess;
    l.busy[b] = false;
    return hipEventSynchronize(l.ev[b]);
}

// Memory that the runtime knows (pinned, managed, on a device) needs no buffer.
static bool unpinned(const void *host)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, host) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

hipError_t HostStage::upload(int device, void *dev, const void *host, size_t bytes, hipStream_t st)
{
    hipError_t e = hipSetDevice(device);
    if (e != hipSuccess)
        return e;
    if (bytes > kMaxUpload || !unpinned(host)) {
        e = hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st);
        return e == hipSuccess ? hipStreamSynchronize(st) : e;
    }
    std::lock_guard<std::mutex> lock(mu_);
    Lane *l = nullptr;
    e = lane(0, &l);
    if (e != hipSuccess)
        return e;
    const unsigned b = l->next++ % kBufs;
    e = wait(*l, b);
    if (e != hipSuccess)
        return e;
    char *buf = l->buf + b * kMaxPiece;
    std::memcpy(buf, host, bytes);
    e = hipMemcpyAsync(dev, buf, bytes, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) {
        l->busy[b] = true;
        e = hipEventRecord(l->ev[b], st);
    }
    return e;
}

struct HostStage::Fetch {
    int device;
    char *host;
    const char *dev;
    size_t bytes, nblocks, piece;
    hipStream_t st;
    BlockKey *keys;
    bool direct; // into host memory itself
    std::atomic<size_t> next{0}; // block to be claimed
};

// One thread's share of a download: blocks claimed one after the other, kBufs pieces on their
// way at a time.
hipError_t HostStage::fetch(Lane &l, Fetch &f)
{
    struct Piece {
        size_t off, len, block;
        bool last; // of its block
    } q[kBufs];
    size_t issued = 0, taken = 0;
    size_t at = 0, end = 0, block = 0; // what of the claimed block is not issued yet
    bool more = true;
    KeyMaker maker;
    hipError_t e = hipSetDevice(f.device);
    for (;;) {
        while (e == hipSuccess && more && issued - taken < kBufs) {
            if (at == end) {
                block = f.next.fetch_add(1, std::memory_order_relaxed);
                if (block >= f.nblocks) {
                    more = false;
                    break;
                }
                at = block * kKeyBlockBytes;
                end = std::min(f.bytes, at + kKeyBlockBytes);
            }
            const unsigned b = (unsigned)(issued % kBufs);
            Piece &p = q[b];
            p.off = at, p.len = std::min(f.piece, end - at), p.block = block;
            at += p.len;
            p.last = at == end;
            e = wait(l, b);
            if (e == hipSuccess)
                e = hipMemcpyAsync(f.direct ? f.host + p.off : l.buf + b * kMaxPiece, f.dev + p.off, p.len,
                                   hipMemcpyDeviceToHost, f.st);
            if (e == hipSuccess) {
                l.busy[b] = true;
                e = hipEventRecord(l.ev[b], f.st);
            }
            ++issued;
        }
        if (e != hipSuccess || issued == taken)
            return e;
        const unsigned b = (unsigned)(taken % kBufs);
        const Piece &p = q[b];
        e = wait(l, b);
        if (e != hipSuccess)
            return e;
        char *to = f.host + p.off;
        const char *from = l.buf + b * kMaxPiece;
        if (f.keys) {
            const size_t whole = p.len / kKeyChunk * kKeyChunk;
            if (f.direct) {
                maker.update(to, whole);
            } else {
                maker.update_copy(to, from, whole);
                std::memcpy(to + whole, from + whole, p.len - whole);
            }
            if (p.last) {
                f.keys[p.block] = maker.finish(to + whole, p.len - whole);
                maker = KeyMaker();
            }
        } else if (!f.direct) {
            stream_copy(to, from, p.len);
        }
        ++taken;
    }
}

hipError_t HostStage::download(int device, void *host, const void *dev, size_t bytes, hipStream_t st,
                               BlockKey *keys, unsigned threads)
{
    if (bytes == 0)
        return hipSuccess;
    std::lock_guard<std::mutex> lock(mu_);
    Fetch f;
    f.device = device;
    f.host = static_cast<char *>(host);
    f.dev = static_cast<const char *>(dev);
    f.bytes = bytes;
    f.nblocks = (bytes + kKeyBlockBytes - 1) / kKeyBlockBytes;
    f.piece = kMinPiece;
    while (f.piece < kMaxPiece && f.piece * (f.piece < ((size_t)1 << 20) ? 4 : 8) < bytes)
        f.piece *= 2;
    f.st = st;
    f.keys = keys;
    f.direct = !unpinned(host);
    threads = (unsigned)std::min<size_t>(std::min(std::max(1u, threads), kMaxLanes), f.nblocks);
    std::vector<Lane *> lanes(threads);
    for (unsigned t = 0; t < threads; ++t) {
        const hipError_t e = lane(t, &lanes[t]);
        if (e != hipSuccess && t == 0)
            return e;
        if (e != hipSuccess) { // fewer threads then
            (void)hipGetLastError();
            lanes.resize(t);
            break;
        }
    }
    std::vector<hipError_t> rc(lanes.size(), hipSuccess);
    struct Pool {
        std::vector<std::thread> threads;
        ~Pool()
        {
            for (std::thread &t : threads)
                if (t.joinable())
                    t.join();
        }
    };
    {
        Pool pool;
        try {
            pool.threads.reserve(lanes.size());
            for (size_t t = 1; t < lanes.size(); ++t)
                pool.threads.emplace_back([&, t] { rc[t] = fetch(*lanes[t], f); });
        } catch (const std::system_error &) {
            // no more threads to be had: those that started and this one share the blocks
        }
        rc[0] = fetch(*lanes[0], f);
    }
    for (const hipError_t e : rc)
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(st); // nothing arrives after the call
            return e;
        }
    return hipSuccess;
}

} // namespace spc3d
