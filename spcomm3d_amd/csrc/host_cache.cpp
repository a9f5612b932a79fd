// Content keys of host operands and copies of host memory (see host_cache.h).  Host code only.
#include "host_cache.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

#if defined(__x86_64__)
#include <immintrin.h>
#endif

namespace spc3d {

namespace {

constexpr int kLanes = 8;                                   // streams of 8-byte words
constexpr int kStripes = (int)(kKeyChunk / (8 * kLanes));   // of a chunk

// Two constants per word of a chunk, one per NH sum.
struct NhKeys {
    alignas(64) uint64_t k[2][kStripes][kLanes];
    constexpr NhKeys() : k()
    {
        uint64_t x = 0x243F6A8885A308D3ull; // splitmix64 from pi's fraction
        for (auto &set : k)
            for (auto &stripe : set)
                for (uint64_t &v : stripe) {
                    x += 0x9E3779B97F4A7C15ull;
                    uint64_t z = x;
                    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
                    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
                    v = z ^ (z >> 31);
                }
    }
};
constexpr NhKeys kNh;

// Between chunks: a bijection of the chained sum (so that nothing a chunk told apart is lost)
// that does not commute with the additions (so that the order of the chunks counts).
constexpr uint64_t kChainXor = 0x452821E638D01377ull, kChainMul = 0x9E3779B1ull;
inline uint64_t chain(uint64_t x) { return (x ^ (x >> 41) ^ kChainXor) * kChainMul; }

inline uint64_t add_halves(uint64_t w, uint64_t k)
{
    return (uint64_t)((uint32_t)w + (uint32_t)k) | (uint64_t)((uint32_t)(w >> 32) + (uint32_t)(k >> 32)) << 32;
}
inline uint64_t product_of_halves(uint64_t x) { return (x & 0xFFFFFFFFu) * (x >> 32); }

void chunks_plain(const unsigned char *p, size_t chunks, uint64_t *a, uint64_t *b, uint64_t *s)
{
    for (size_t c = 0; c < chunks; ++c, p += kKeyChunk) {
        for (int t = 0; t < kStripes; ++t)
            for (int l = 0; l < kLanes; ++l) {
                uint64_t w;
                std::memcpy(&w, p + (size_t)(t * kLanes + l) * 8, 8);
                a[l] += product_of_halves(add_halves(w, kNh.k[0][t][l]));
                b[l] += product_of_halves(add_halves(w, kNh.k[1][t][l]));
                s[l] += w;
            }
        for (int l = 0; l < kLanes; ++l)
            a[l] = chain(a[l]), b[l] = chain(b[l]);
    }
}

#if defined(__x86_64__)
__attribute__((target("avx2"))) inline __m256i chain_avx2(__m256i x)
{
    x = _mm256_xor_si256(_mm256_xor_si256(x, _mm256_srli_epi64(x, 41)), _mm256_set1_epi64x((long long)kChainXor));
    const __m256i m = _mm256_set1_epi64x((long long)kChainMul);
    const __m256i hi = _mm256_mul_epu32(_mm256_srli_epi64(x, 32), m);
    return _mm256_add_epi64(_mm256_mul_epu32(x, m), _mm256_slli_epi64(hi, 32));
}

// COPY: every vector read is also stored to `to` (32-byte aligned), past the caches.
template <bool COPY>
__attribute__((target("avx2"))) void chunks_avx2(const unsigned char *p, unsigned char *to, size_t chunks,
                                                 uint64_t *a, uint64_t *b, uint64_t *s)
{
    __m256i A[2], B[2], S[2];
    for (int h = 0; h < 2; ++h) {
        A[h] = _mm256_load_si256((const __m256i *)a + h);
        B[h] = _mm256_load_si256((const __m256i *)b + h);
        S[h] = _mm256_load_si256((const __m256i *)s + h);
    }
    for (size_t c = 0; c < chunks; ++c, p += kKeyChunk, to += COPY ? kKeyChunk : 0) {
        for (int t = 0; t < kStripes; ++t)
            for (int h = 0; h < 2; ++h) {
                const __m256i w = _mm256_loadu_si256((const __m256i *)(p + t * 64 + h * 32));
                const __m256i x = _mm256_add_epi32(w, _mm256_load_si256((const __m256i *)kNh.k[0][t] + h));
                const __m256i y = _mm256_add_epi32(w, _mm256_load_si256((const __m256i *)kNh.k[1][t] + h));
                A[h] = _mm256_add_epi64(A[h], _mm256_mul_epu32(x, _mm256_srli_epi64(x, 32)));
                B[h] = _mm256_add_epi64(B[h], _mm256_mul_epu32(y, _mm256_srli_epi64(y, 32)));
                S[h] = _mm256_add_epi64(S[h], w);
                if (COPY)
                    _mm256_stream_si256((__m256i *)(to + t * 64 + h * 32), w);
            }
        for (int h = 0; h < 2; ++h)
            A[h] = chain_avx2(A[h]), B[h] = chain_avx2(B[h]);
    }
    for (int h = 0; h < 2; ++h) {
        _mm256_store_si256((__m256i *)a + h, A[h]);
        _mm256_store_si256((__m256i *)b + h, B[h]);
        _mm256_store_si256((__m256i *)s + h, S[h]);
    }
    if (COPY)
        _mm_sfence();
}

__attribute__((target("avx2"))) void stream_copy_avx2(unsigned char *to, const unsigned char *from, size_t bytes)
{
    const size_t head = std::min<size_t>(bytes, (32 - ((uintptr_t)to & 31)) & 31);
    std::memcpy(to, from, head);
    to += head, from += head, bytes -= head;
    size_t i = 0;
    for (; i + 128 <= bytes; i += 128) {
        const __m256i v0 = _mm256_loadu_si256((const __m256i *)(from + i));
        const __m256i v1 = _mm256_loadu_si256((const __m256i *)(from + i + 32));
        const __m256i v2 = _mm256_loadu_si256((const __m256i *)(from + i + 64));
        const __m256i v3 = _mm256_loadu_si256((const __m256i *)(from + i + 96));
        _mm256_stream_si256((__m256i *)(to + i), v0);
        _mm256_stream_si256((__m256i *)(to + i + 32), v1);
        _mm256_stream_si256((__m256i *)(to + i + 64), v2);
        _mm256_stream_si256((__m256i *)(to + i + 96), v3);
    }
    _mm_sfence();
    std::memcpy(to + i, from + i, bytes - i);
}

bool have_avx2()
{
    static const bool yes = __builtin_cpu_supports("avx2");
    return yes;
}
#else
bool have_avx2() { return false; }
#endif

} // namespace

KeyMaker::KeyMaker(bool portable) : vector_(!portable && have_avx2())
{
    for (int l = 0; l < kLanes; ++l) {
        a_[l] = kNh.k[1][0][l] * 3;
        b_[l] = kNh.k[0][1][l] * 5;
        s_[l] = 0;
    }
}

void KeyMaker::update(const void *data, size_t bytes)
{
    const unsigned char *p = static_cast<const unsigned char *>(data);
    total_ += bytes;
#if defined(__x86_64__)
    if (vector_) {
        chunks_avx2<false>(p, nullptr, bytes / kKeyChunk, a_, b_, s_);
        return;
    }
#endif
    chunks_plain(p, bytes / kKeyChunk, a_, b_, s_);
}

void KeyMaker::update_copy(void *to, const void *from, size_t bytes)
{
#if defined(__x86_64__)
    if (vector_ && ((uintptr_t)to & 31) == 0) {
        total_ += bytes;
        chunks_avx2<true>(static_cast<const unsigned char *>(from), static_cast<unsigned char *>(to),
                          bytes / kKeyChunk, a_, b_, s_);
        return;
    }
#endif
    // a few chunks at a time, so that the second read finds them in the first-level cache
    const unsigned char *p = static_cast<const unsigned char *>(from);
    unsigned char *q = static_cast<unsigned char *>(to);
    for (size_t i = 0; i < bytes; i += 16 * kKeyChunk) {
        const size_t n = std::min(16 * kKeyChunk, bytes - i);
        std::memcpy(q + i, p + i, n);
        update(p + i, n);
    }
}

BlockKey KeyMaker::finish(const void *data, size_t bytes)
{
    const size_t whole = bytes / kKeyChunk * kKeyChunk;
    if (whole)
        update(data, whole);
    if (bytes > whole) { // the last chunk, filled up with zeros; the length counts below
        unsigned char last[kKeyChunk] = {0};
        std::memcpy(last, static_cast<const unsigned char *>(data) + whole, bytes - whole);
        update(last, kKeyChunk);
        total_ -= kKeyChunk - (bytes - whole);
    }
    BlockKey k;
    k.nh0 = total_, k.nh1 = ~total_;
    for (int l = 0; l < kLanes; ++l) {
        k.nh0 = chain(k.nh0 + a_[l]);
        k.nh1 = chain(k.nh1 + b_[l]);
        k.sum += s_[l];
        k.fold = chain(k.fold + s_[l]);
    }
    return k;
}

BlockKey key_of_block_portable(const void *data, size_t bytes) { return KeyMaker(true).finish(data, bytes); }

BlockKey key_of_block(const void *data, size_t bytes) { return KeyMaker().finish(data, bytes); }

void stream_copy(void *to, const void *from, size_t bytes)
{
#if defined(__x86_64__)
    if (have_avx2()) {
        stream_copy_avx2(static_cast<unsigned char *>(to), static_cast<const unsigned char *>(from), bytes);
        return;
    }
#endif
    std::memcpy(to, from, bytes);
}

void keys_of(const void *data, size_t bytes, std::vector<BlockKey> &out, unsigned threads)
{
    const size_t nblocks = (bytes + kKeyBlockBytes - 1) / kKeyBlockBytes;
    out.assign(nblocks, BlockKey());
    if (nblocks == 0)
        return;
    if (threads == 0) {
        const unsigned hw = std::thread::hardware_concurrency();
        threads = std::min(8u, hw ? hw : 1u);
    }
    threads = (unsigned)std::min<size_t>(threads, nblocks);
    const unsigned char *p = static_cast<const unsigned char *>(data);
    std::atomic<size_t> next{0};
    auto work = [&]() {
        for (;;) {
            const size_t b = next.fetch_add(1, std::memory_order_relaxed);
            if (b >= nblocks)
                return;
            const size_t off = b * kKeyBlockBytes;
            out[b] = key_of_block(p + off, std::min(kKeyBlockBytes, bytes - off));
        }
    };
    if (threads <= 1) {
        work();
        return;
    }
    std::vector<std::thread> pool;
    pool.reserve(threads - 1);
    try {
        for (unsigned t = 1; t < threads; ++t)
            pool.emplace_back(work);
    } catch (const std::system_error &) {
        // no more threads to be had: those that started and this one share the blocks
    }
    work();
    for (std::thread &t : pool)
        t.join();
}

} // namespace spc3d
