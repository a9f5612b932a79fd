// Copies between pageable host memory and the device through pinned buffers of the context.
//
// The runtime's own copies of pageable memory run at 29 GB/s up and 17 GB/s down on this host;
// small ones pay its staging (0.25 MiB: 110 us).  A pinned buffer moves at 57 GB/s and a core
// copies at 30 to 40, so a download goes through pinned buffers in pieces, the next ones on their
// way while the CPU copies one, and is keyed by the copy that brings it to the caller's memory
// (KeyMaker).  64 MiB down: 3.8 -> 1.7 ms; 1 MiB the same 0.06; 64 KiB: 36 -> 18 us.
// An upload has nothing to overlap with but the copy itself: above 512 KiB the runtime, which
// pins the caller's pages, is as fast, and only smaller ones take a buffer (0.25 MiB: 25 us).
//
// The pinned memory is allocated by the first transfer that uses it (1.5 MiB for small ones, 12 MiB
// per host thread that takes part in a large one) and freed with the context or its host-call cache.
// Without it (the host's pinned memory is used up) transfers go the runtime's own way, slower.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <memory>
#include <mutex>
#include <vector>

#include "host_cache.h"

namespace spc3d {

class HostStage {
  public:
    HostStage() = default;
    HostStage(const HostStage &) = delete;
    HostStage &operator=(const HostStage &) = delete;
    ~HostStage() { release(); }

    // Queues dev = host on `st` and returns when `host` has been read.  May be called by
    // two threads at once.
    hipError_t upload(int device, void *dev, const void *host, size_t bytes, hipStream_t st);
    // host = dev after what is queued on `st`; returns when it is there.  keys (null: none): those
    // of host's kKeyBlockBytes blocks.  On up to `threads` threads, the caller's included.
    hipError_t download(int device, void *host, const void *dev, size_t bytes, hipStream_t st,
                        BlockKey *keys, unsigned threads);
    void release();

  private:
    // A piece costs 11 us beside the copy itself, and what cannot overlap is one piece's way
    // down and one's copy: a quarter of the transfer for pieces up to 1 MiB, an eighth above (a
    // power of two, so that pieces divide the key blocks).
    static constexpr size_t kMinPiece = (size_t)1 << 19, kMaxPiece = kKeyBlockBytes;
    static constexpr unsigned kBufs = 3, kMaxLanes = 8;
    static constexpr size_t kMaxUpload = (size_t)1 << 19; // through a buffer
    struct Lane { // the buffers of one thread
        char *buf = nullptr;
        size_t piece = 0; // bytes of one of them: kMinPiece or kMaxPiece
        hipEvent_t ev[kBufs] = {};
        bool busy[kBufs] = {}; // a copy out of (into) the buffer may be under way
        unsigned next = 0;
    };
    // Thread i's buffers, for pieces of `piece` bytes (or less, when there is only memory for
    // kMinPiece).  Null: there is none.
    Lane *lane(unsigned i, size_t piece);
    static hipError_t wait(Lane &l, unsigned b);
    struct Fetch;
    static hipError_t fetch(Lane &l, Fetch &f);
    static hipError_t fetch_unstaged(Fetch &f);
    std::mutex mu_;
    std::vector<std::unique_ptr<Lane>> lanes_;
};

} // namespace spc3d
