// Copies between pageable host memory and the device (see host_stage.h).
#include "host_stage.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <new>
#include <thread>

namespace spc3d {

HostStage::Lane *HostStage::lane(unsigned i, size_t piece)
{
    piece = piece > kMinPiece ? kMaxPiece : kMinPiece;
    try {
        lanes_.reserve(kMaxLanes);
        while (lanes_.size() <= i) {
            std::unique_ptr<Lane> l(new Lane());
            hipError_t e = hipSuccess;
            for (unsigned b = 0; b < kBufs && e == hipSuccess; ++b)
                e = hipEventCreateWithFlags(&l->ev[b], hipEventDisableTiming);
            if (e != hipSuccess) {
                (void)hipGetLastError();
                for (hipEvent_t ev : l->ev)
                    if (ev) (void)hipEventDestroy(ev);
                return nullptr;
            }
            lanes_.push_back(std::move(l));
        }
    } catch (const std::bad_alloc &) {
        return nullptr;
    }
    Lane &l = *lanes_[i];
    for (; l.piece < piece; piece = kMinPiece) {
        char *buf = nullptr;
        if (hipHostMalloc((void **)&buf, piece * kBufs, hipHostMallocDefault) == hipSuccess) {
            for (unsigned b = 0; b < kBufs; ++b)
                (void)wait(l, b);
            if (l.buf)
                (void)hipHostFree(l.buf);
            l.buf = buf;
            l.piece = piece;
            break;
        }
        (void)hipGetLastError();
        if (piece == kMinPiece)
            break;
    }
    return l.buf ? &l : nullptr;
}

void HostStage::release()
{
    std::lock_guard<std::mutex> lock(mu_);
    for (auto &l : lanes_) {
        for (unsigned b = 0; b < kBufs; ++b) {
            (void)wait(*l, b);
            (void)hipEventDestroy(l->ev[b]);
        }
        if (l->buf)
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
    if (bytes <= kMaxUpload && unpinned(host)) {
        std::lock_guard<std::mutex> lock(mu_);
        if (Lane *l = lane(0, kMinPiece)) {
            const unsigned b = l->next++ % kBufs;
            e = wait(*l, b);
            if (e != hipSuccess)
                return e;
            char *buf = l->buf + b * l->piece;
            std::memcpy(buf, host, bytes);
            e = hipMemcpyAsync(dev, buf, bytes, hipMemcpyHostToDevice, st);
            if (e == hipSuccess) {
                l->busy[b] = true;
                e = hipEventRecord(l->ev[b], st);
            }
            return e;
        }
    }
    e = hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
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
                e = hipMemcpyAsync(f.direct ? f.host + p.off : l.buf + b * l.piece, f.dev + p.off, p.len,
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
        const char *from = l.buf + b * l.piece;
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

// A whole download by the runtime's own copy, keyed where it arrived.
hipError_t HostStage::fetch_unstaged(Fetch &f)
{
    hipError_t e = hipSetDevice(f.device);
    if (e == hipSuccess)
        e = hipMemcpyAsync(f.host, f.dev, f.bytes, hipMemcpyDeviceToHost, f.st);
    if (e == hipSuccess)
        e = hipStreamSynchronize(f.st);
    for (size_t b = 0; e == hipSuccess && f.keys && b < f.nblocks; ++b)
        f.keys[b] = key_of_block(f.host + b * kKeyBlockBytes,
                                 std::min(kKeyBlockBytes, f.bytes - b * kKeyBlockBytes));
    return e;
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
    Lane *lanes[kMaxLanes] = {};
    unsigned n = 0;
    for (; n < threads; ++n) { // fewer threads when there is no memory for more
        lanes[n] = lane(n, f.piece);
        if (!lanes[n])
            break;
        f.piece = std::min(f.piece, lanes[n]->piece);
    }
    if (n == 0)
        return fetch_unstaged(f);
    hipError_t rc[kMaxLanes];
    std::fill(rc, rc + kMaxLanes, hipSuccess);
    struct Pool {
        std::thread threads[kMaxLanes];
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
            for (unsigned t = 1; t < n; ++t)
                pool.threads[t] = std::thread([&, t] { rc[t] = fetch(*lanes[t], f); });
        } catch (const std::exception &) {
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
