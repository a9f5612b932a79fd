// Content keys of host operands, for the one-shot entry points over host memory
// (spc3d_sddmm_host / spc3d_spmm_host).  The reference's drivers call the kernel several
// times over one pattern and the same dense panels (miniapp/bench_both.cpp:202-203,
// bench_spmm.cpp:185-186), and rewrite indices in place at the same addresses between
// groups of calls (ReMapIndices, bench_both.cpp:200-205): what a call may reuse from the
// one before is decided by what the operands hold, never by where they are.
//
// An operand is keyed block by block (4 MiB): a block whose key is unchanged is not sent
// again, a changed one is.  Every byte goes into the key, over several threads (reading
// host memory with a few threads is faster than sending it: the point of the exercise).
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

namespace spc3d {

// Key of one block: two NH sums (UMAC's universal hash: of every 8-byte word, the product of
// its halves after a 32-bit addition of a position's constant to each) chained over chunks of
// 1 KiB, the words' plain sum, and the sums of the eight interleaved streams of words folded
// together.  A change of one word always changes the sum; several changes have to cancel in
// the sum, the streams' sums and both chains at once.
struct BlockKey {
    uint64_t nh0 = 0, nh1 = 0, sum = 0, fold = 0;
    bool operator==(const BlockKey &o) const
    {
        return nh0 == o.nh0 && nh1 == o.nh1 && sum == o.sum && fold == o.fold;
    }
    bool operator!=(const BlockKey &o) const { return !(*this == o); }
};

constexpr size_t kKeyBlockBytes = (size_t)4 << 20;
constexpr size_t kKeyChunk = 1024;

// A key made piece by piece: update() over whole chunks (any number of them), then finish() over
// the rest of the block.  Bound by the read of the memory: 46 GB/s on one core of an EPYC host
// whose plain sum over the same memory runs at 49 (the CRC-32C streams this replaced: 30).
class KeyMaker {
  public:
    explicit KeyMaker(bool portable = false);
    void update(const void *data, size_t bytes);                 // bytes % kKeyChunk == 0
    void update_copy(void *to, const void *from, size_t bytes);  // the same, and to = from
    BlockKey finish(const void *data, size_t bytes);             // what is left, any length
  private:
    alignas(64) uint64_t a_[8], b_[8], s_[8];
    uint64_t total_ = 0;
    bool vector_;
};

BlockKey key_of_block(const void *data, size_t bytes);
// The form used on hosts without AVX2 (the same keys, word by word); exposed so that it is
// tested on hosts that have it.
BlockKey key_of_block_portable(const void *data, size_t bytes);

// Keys of every kKeyBlockBytes block of `data` (the last one may be short), computed on up
// to `threads` threads (0: a default from the machine, at most 8).
void keys_of(const void *data, size_t bytes, std::vector<BlockKey> &out, unsigned threads = 0);

// to = from without leaving `to` in the caches (it is read next by a device, or is larger than
// they are); any alignment.
void stream_copy(void *to, const void *from, size_t bytes);

} // namespace spc3d
