// Device-side plan construction (see plan_device.h).  Every step restates one
// step of build_host_plan (plan_host.cpp) with a parallel primitive that gives
// the same result: histograms by atomics, prefix sums by device scans, the
// stable counting sorts by stable radix sorts.
#include "plan_device.h"

#include <hip/hip_runtime.h>
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include <algorithm>
#include <cstdio>
#include <initializer_list>

#include "../../include/spcomm3d_hip.h"

namespace spc3d {
namespace {

constexpr int kTB = 256;

struct Counters { // one device-resident block, zeroed (first_bad: all ones) before use
    uint32_t first_bad;
    uint32_t rows_touched, max_row, cols_touched, max_cdeg;
    uint32_t not_identity;
    uint32_t qcount[kSlices], qlong[kSlices];
    uint32_t nlong;
    uint32_t rows_unsorted, cols_unsorted;
    uint32_t row_changes; // entries whose row is not their predecessor's
    unsigned long long covered;
    unsigned long long row_sq;
    unsigned long long load[kSlices], any_load, pref_load[kSlices];
    unsigned long long hot_weight[kHotClasses];
};

// Owning device buffer; back to the pool on scope exit unless released.
template <typename T> struct DBuf {
    T *p = nullptr;
    DBuf() = default;
    DBuf(const DBuf &) = delete;
    DBuf &operator=(const DBuf &) = delete;
    ~DBuf() { reset(); }
    void reset()
    {
        if (p)
            pool_->put(p);
        p = nullptr;
    }
    hipError_t alloc(const DevStream &st, size_t count)
    {
        reset();
        pool_ = st.pool;
        return pool_->get((void **)&p, count * sizeof(T));
    }
    T *release()
    {
        T *r = p;
        p = nullptr;
        return r;
    }

  private:
    DevPool *pool_ = nullptr;
};

// Scratch device memory of one call: a few large blocks of the pool, handed out front to
// back and given back together when the call returns.
class Arena {
  public:
    explicit Arena(const DevStream &st) : pool_(*st.pool) {}
    Arena(const Arena &) = delete;
    Arena &operator=(const Arena &) = delete;
    ~Arena()
    {
        for (int i = 0; i < nblocks_; ++i)
            pool_.put(blocks_[i]);
    }
    // Makes sure that the next `bytes` come out of one block.
    hipError_t reserve(size_t bytes)
    {
        if (bytes <= left_)
            return hipSuccess;
        if (nblocks_ == kMaxBlocks)
            return hipErrorOutOfMemory;
        void *b = nullptr;
        // Up to twice as large a kept block does: plans of one program need scratch of a few sizes, by the order of
        // their entries, and it goes back at once (a column-sorted pattern of 84 M entries and its companion, whose
        // rows come in order, kept both sizes and ran past the pool's limit: 16.2 ms, 15.7 with one).
        const hipError_t e = pool_.get(&b, bytes, bytes);
        if (e != hipSuccess)
            return e;
        blocks_[nblocks_++] = b;
        cur_ = static_cast<char *>(b);
        left_ = bytes;
        return hipSuccess;
    }
    hipError_t take(void **p, size_t bytes)
    {
        *p = nullptr;
        if (bytes == 0)
            return hipSuccess;
        bytes = (bytes + 255) / 256 * 256;
        const hipError_t e = reserve(bytes > left_ && bytes < kMinBlock ? kMinBlock : bytes);
        if (e != hipSuccess)
            return e;
        *p = cur_;
        cur_ += bytes;
        left_ -= bytes;
        return hipSuccess;
    }

  private:
    static constexpr int kMaxBlocks = 64;
    static constexpr size_t kMinBlock = (size_t)4 << 20;
    DevPool &pool_;
    void *blocks_[kMaxBlocks] = {};
    int nblocks_ = 0;
    char *cur_ = nullptr;
    size_t left_ = 0;
};

// An array in the arena; nothing to free.
template <typename T> struct SBuf {
    T *p = nullptr;
    hipError_t alloc(Arena &a, size_t count)
    {
        return a.take(reinterpret_cast<void **>(&p), count * sizeof(T));
    }
};

inline uint32_t grid_for(uint64_t n)
{
    const uint64_t want = (n + kTB - 1) / kTB;
    const uint64_t cap = 256 * 32;
    return (uint32_t)(want < 1 ? 1 : (want > cap ? cap : want));
}

inline uint32_t small_grid_for(uint64_t n) // kernels that end in one atomic per workgroup
{
    const uint32_t g = grid_for(n);
    return g > 1024 ? 1024 : g;
}

// Kernels that end in a dozen and more atomics per workgroup: ten nanoseconds each, one after the
// other (17 sums over 700 k pieces: 100 us on 1,024 workgroups).
inline uint32_t few_grid_for(uint64_t n)
{
    const uint32_t g = grid_for(n);
    return g > 192 ? 192 : g;
}

inline int bits_for(uint64_t max_value) // bits needed to hold max_value (at least 1)
{
    int b = 1;
    while (b < 64 && (max_value >> b) != 0)
        ++b;
    return b;
}

#define GRID_STRIDE(i, n)                                                                         \
    for (uint64_t i = (uint64_t)blockIdx.x * kTB + threadIdx.x; i < (n);                         \
         i += (uint64_t)gridDim.x * kTB)

template <typename T> __device__ __forceinline__ T wave_sum(T v)
{
    for (int s = 32; s >= 1; s >>= 1)
        v += __shfl_xor(v, s, 64);
    return v;
}

// Sum (maximum) of v over the workgroup, valid in thread 0; every thread of the
// workgroup calls.  The kernels that count into the Counters block add one value
// per workgroup and run on a small grid: device-wide atomics on a handful of
// addresses are served one after the other, and one per wavefront of a full-size
// grid cost more than the rest of the kernel.
template <typename T> __device__ __forceinline__ T block_sum(T v)
{
    __shared__ T part[kTB / 64];
    v = wave_sum(v);
    __syncthreads(); // an earlier call's part[] has been read
    if ((threadIdx.x & 63) == 0)
        part[threadIdx.x >> 6] = v;
    __syncthreads();
    T t = 0;
    if (threadIdx.x == 0)
        for (int w = 0; w < kTB / 64; ++w)
            t += part[w];
    return t;
}
__device__ __forceinline__ uint32_t block_max(uint32_t v)
{
    __shared__ uint32_t part[kTB / 64];
    for (int s = 32; s >= 1; s >>= 1) {
        const uint32_t o = __shfl_xor(v, s, 64);
        v = v > o ? v : o;
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
        part[threadIdx.x >> 6] = v;
    __syncthreads();
    uint32_t t = 0;
    if (threadIdx.x == 0)
        for (int w = 0; w < kTB / 64; ++w)
            t = t > part[w] ? t : part[w];
    return t;
}

template <typename T> __global__ void fill_k(T *p, uint64_t n, T v)
{
    GRID_STRIDE(i, n) p[i] = v;
}

__global__ void iota_k(uint32_t *p, uint64_t n)
{
    GRID_STRIDE(i, n) p[i] = (uint32_t)i;
}

// Adds 1 to cnt[key] for every lane with a valid key, with one atomic per run of
// equal keys in consecutive lanes (sorted COO puts a whole wavefront on one row,
// and same-address atomics of a wavefront are served one after the other).
__device__ __forceinline__ void count_runs(uint32_t *cnt, uint32_t key, bool valid)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t prev = __shfl_up(key, 1, 64);
    const bool prev_valid = __shfl_up((int)valid, 1, 64) != 0;
    const bool head = valid && (lane == 0 || !prev_valid || prev != key);
    // a run ends where the next head starts or where the keys stop being valid
    const unsigned long long stops = __ballot(head || !valid);
    if (head) {
        const unsigned long long above = lane == 63 ? 0ull : stops >> (lane + 1);
        const uint32_t len = above ? (uint32_t)__ffsll((long long)above) : 64u - lane;
        atomicAdd(cnt + key, len);
    }
}

// The first out-of-range entry, if any; whether the rows, and the columns, ever step down; how often
// the row changes.  Four
// entries of a thread in flight (16 M entries: 62 us with one, now 42).
__global__ void check_k(const uint32_t *__restrict__ ii, const uint32_t *__restrict__ jj,
                        uint64_t nnz, uint32_t nrows, uint32_t ncols, Counters *C)
{
    uint32_t bad = 0xFFFFFFFFu;
    bool down = false, cdown = false;
    uint32_t changes = 0;
    const uint64_t stride = (uint64_t)gridDim.x * kTB;
    for (uint64_t e = (uint64_t)blockIdx.x * kTB + threadIdx.x; e < nnz; e += 4 * stride) {
        uint32_t at[4], r[4], c[4], rp[4], cp[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            at[u] = (uint32_t)(e + u * stride < nnz ? e + u * stride : e);
            const uint32_t before = at[u] ? at[u] - 1 : 0;
            r[u] = ii[at[u]];
            c[u] = jj[at[u]];
            rp[u] = ii[before];
            cp[u] = jj[before];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if ((r[u] >= nrows || c[u] >= ncols) && at[u] < bad)
                bad = at[u];
            down |= rp[u] > r[u];
            changes += e + u * stride < nnz && rp[u] != r[u];
            cdown |= cp[u] > c[u];
        }
    }
    if (bad != 0xFFFFFFFFu)
        atomicMin(&C->first_bad, bad); // rare: the build fails
    changes = block_sum(changes);
    if (threadIdx.x == 0 && changes)
        atomicAdd(&C->row_changes, changes);
    down = __syncthreads_or(down);
    cdown = __syncthreads_or(cdown);
    if (threadIdx.x == 0 && down)
        atomicOr(&C->rows_unsorted, 1u);
    if (threadIdx.x == 0 && cdown)
        atomicOr(&C->cols_unsorted, 1u);
}

// Row histogram of entries that come in runs of a row: whole wavefronts walk the entries
// together and pool their counts, one atomic per run of equal rows.
__global__ void hist_sorted_k(const uint32_t *__restrict__ ii, uint64_t nnz, uint32_t *rowcnt)
{
    const uint64_t stride = (uint64_t)gridDim.x * kTB;
    for (uint64_t base = (uint64_t)blockIdx.x * kTB + (threadIdx.x & ~63u); base < nnz;
         base += stride) {
        const uint64_t e = base + (threadIdx.x & 63u);
        const bool ok = e < nnz;
        count_runs(rowcnt, ok ? ii[e] : 0u, ok);
    }
}

// Histogram from sorted ids, where there are any: where a run of equal ids starts, its position goes to
// start[id]; where it ends, the position after it goes to deg[id] (zeroed before); deg[id] -= start[id]
// then leaves the run's length.  The ids were checked against nbins before.
__global__ void run_bounds_k(const uint32_t *__restrict__ sorted, uint64_t n, uint32_t nbins,
                             uint32_t *start, uint32_t *deg)
{
    GRID_STRIDE(i, n)
    {
        const uint32_t k = sorted[i];
        if (k >= nbins)
            continue;
        if (i == 0 || sorted[i - 1] != k)
            start[k] = (uint32_t)i;
        if (i + 1 == n || sorted[i + 1] != k)
            deg[k] = (uint32_t)(i + 1);
    }
}
__global__ void run_lengths_k(const uint32_t *__restrict__ start, uint64_t nbins, uint32_t *deg)
{
    GRID_STRIDE(c, nbins)
    {
        const uint32_t end = deg[c];
        if (end)
            deg[c] = end - start[c];
    }
}

// How often every id comes (count_ids): the ids lie in buckets of 1 << low by their upper bits, which are cut
// into parts of at most `part` entries; a workgroup counts a part in LDS.
constexpr int kCountTB = 1024;

// The first of n keys, ascending in key >> low, that is `bucket` or above there.  By a wavefront, 64 probes at a time.
__device__ __forceinline__ uint32_t bucket_start(const uint32_t *__restrict__ key, uint32_t n, uint32_t low,
                                                 uint32_t bucket)
{
    uint32_t lo = 0, len = n; // the answer is in [lo, lo + len]
    while (len) {
        const uint32_t step = len / 64 + 1, lane = threadIdx.x & 63u;
        const bool in = (uint64_t)lane * step < len;
        const unsigned long long below = __ballot(in && key[lo + (in ? lane * step : 0u)] >> low < bucket);
        const uint32_t k = (uint32_t)__popcll(below); // probes 0 .. k - 1 are below, the others are not
        if (k == 0)
            return lo;
        const uint32_t past = (k - 1) * step + 1; // of lo: at least so much further, and less than a step more
        lo += past;
        len = len - past < step - 1 ? len - past : step - 1;
    }
    return lo;
}
__global__ void bucket_parts_k(const uint32_t *__restrict__ key, uint32_t n, uint32_t low, uint32_t nbuckets,
                               uint32_t part, uint32_t *start, uint32_t *parts)
{
    const uint32_t b = blockIdx.x * (kTB / 64) + threadIdx.x / 64;
    if (b > nbuckets)
        return;
    const uint32_t lo = b < nbuckets ? bucket_start(key, n, low, b) : n;
    const uint32_t hi = b < nbuckets ? bucket_start(key, n, low, b + 1) : n;
    if ((threadIdx.x & 63u) == 0) {
        start[b] = lo;
        parts[b] = parts_of(hi - lo, part);
    }
}
__global__ void __launch_bounds__(kCountTB)
bucket_count_k(const uint32_t *__restrict__ key, const uint32_t *__restrict__ start,
               const uint32_t *__restrict__ first_part, uint32_t low, uint32_t nbuckets, uint32_t part, uint32_t *counts)
{
    __shared__ uint32_t count[1u << kCountBits];
    const uint32_t g = blockIdx.x, mask = (1u << low) - 1;
    if (g >= first_part[nbuckets])
        return;
    uint32_t b = 0, up = nbuckets; // first_part[b] <= g < first_part[up]
    while (up - b > 1) {
        const uint32_t mid = b + (up - b) / 2;
        if (first_part[mid] <= g)
            b = mid;
        else
            up = mid;
    }
    const uint32_t from = start[b] + (g - first_part[b]) * part, left = start[b + 1] - from;
    const uint32_t n = left < part ? left : part;
    for (uint32_t i = threadIdx.x; i <= mask; i += kCountTB)
        count[i] = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += 4 * kCountTB) {
        uint32_t v[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
            v[u] = key[from + (i + u * kCountTB < n ? i + u * kCountTB : i)];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
            if (i + u * kCountTB < n)
                atomicAdd(&count[v[u] & mask], 1u);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i <= mask; i += kCountTB)
        counts[((uint64_t)g << low) + i] = count[i];
}
__global__ void bucket_sum_k(const uint32_t *__restrict__ counts, const uint32_t *__restrict__ first_part,
                             uint32_t low, uint64_t nbins, uint32_t *cnt)
{
    GRID_STRIDE(c, nbins)
    {
        const uint32_t b = (uint32_t)(c >> low), at = (uint32_t)c & ((1u << low) - 1);
        uint32_t sum = 0;
        for (uint32_t g = first_part[b]; g < first_part[b + 1]; ++g)
            sum += counts[((uint64_t)g << low) + at];
        cnt[c] = sum;
    }
}

// Number of non-zero counts, the largest count and, with sq, the sum of count * min(count, 2048).
__global__ void stats_k(const uint32_t *__restrict__ cnt, uint64_t n, uint32_t *touched,
                        uint32_t *maxv, unsigned long long *sq)
{
    uint32_t t = 0, m = 0;
    unsigned long long s = 0;
    const uint64_t stride = (uint64_t)gridDim.x * kTB;
    for (uint64_t i = (uint64_t)blockIdx.x * kTB + threadIdx.x; i < n; i += 4 * stride) {
        uint32_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            v[u] = i + u * stride < n ? cnt[i + u * stride] : 0u;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            t += v[u] != 0;
            m = m > v[u] ? m : v[u];
            s += (unsigned long long)v[u] * (v[u] < 2048 ? v[u] : 2048);
        }
    }
    t = block_sum(t);
    m = block_max(m);
    if (sq)
        s = block_sum(s);
    if (threadIdx.x == 0) {
        if (sq && s)
            atomicAdd(sq, s);
        if (t)
            atomicAdd(touched, t);
        if (m)
            atomicMax(maxv, m);
    }
}

__global__ void sum_first_k(const uint32_t *__restrict__ v, uint64_t n, unsigned long long *out)
{
    unsigned long long s = 0;
    GRID_STRIDE(i, n) s += v[i];
    s = block_sum(s);
    if (threadIdx.x == 0 && s)
        atomicAdd(out, s);
}

// Entries of the n hottest columns by the low bits of the column (hot_rows_crowd); one workgroup.
__global__ void __launch_bounds__(kTB)
hot_weight_k(const uint32_t *__restrict__ order, const uint32_t *__restrict__ deg, uint32_t n,
             unsigned long long *__restrict__ weight)
{
    __shared__ unsigned long long sum[kHotClasses];
    if (threadIdx.x < kHotClasses)
        sum[threadIdx.x] = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += kTB)
        atomicAdd(&sum[order[i] % kHotClasses], (unsigned long long)deg[i]);
    __syncthreads();
    if (threadIdx.x < kHotClasses)
        weight[threadIdx.x] = sum[threadIdx.x];
}

// rank[hot[i]] = i (rank: all ones before)
__global__ void hot_ranks_k(const uint32_t *__restrict__ hot, uint64_t n, uint16_t *__restrict__ rank)
{
    GRID_STRIDE(i, n) rank[hot[i]] = (uint16_t)i;
}
__global__ void encode_hot_k(const uint32_t *__restrict__ col, uint64_t n,
                             const uint16_t *__restrict__ rank, uint32_t *__restrict__ out)
{
    GRID_STRIDE(q, n)
    {
        const uint32_t c = col[q], r = rank[c];
        out[q] = r == 0xFFFFu ? c : kHotRow | r;
    }
}

// Classes of the htot hottest columns (order[] = columns by degree, highest first).
__global__ void classify_k(const uint32_t *__restrict__ order, uint64_t htot, uint32_t hrep,
                           uint8_t *cls)
{
    GRID_STRIDE(i, htot)
    cls[order[i]] = i < hrep ? kClsRep : slice_of_rank(i - hrep);
}

// (bytes: the keys of an unsorted pattern ask for them at random, and 1 M fit an L2 four times)
__global__ void hubflag_k(const uint32_t *__restrict__ rowcnt, uint32_t nrows, uint32_t hub_min,
                          uint8_t *flag)
{
    GRID_STRIDE(r, (uint64_t)nrows + 1) flag[r] = r < nrows && rowcnt[r] >= hub_min;
}

// Per hub row, the number of entries in each of the 9 groups, from the sorted keys (keys_k): where a
// run of equal keys starts its position is taken off the count (zeroed before), where it ends the
// position after it is added.  16 M entries of R-MAT 20: an atomic per group and wavefront of the
// unsorted entries took 244 us, this 49.
template <typename KeyT>
__global__ void hubcount_k(const KeyT *__restrict__ key, uint64_t nnz,
                           const uint8_t *__restrict__ hubflag,
                           const uint32_t *__restrict__ hubpos, uint32_t *hubcnt)
{
    GRID_STRIDE(i, nnz)
    {
        const KeyT k = key[i];
        const bool first = i == 0 || key[i - 1] != k, last = i + 1 == nnz || key[i + 1] != k;
        if (!first && !last)
            continue;
        const uint32_t r = (uint32_t)(k >> 4);
        if (!hubflag[r])
            continue;
        const uint32_t n = (last ? (uint32_t)(i + 1) : 0u) - (first ? (uint32_t)i : 0u);
        atomicAdd(hubcnt + (size_t)hubpos[r] * 9 + (uint32_t)(k & 15), n);
    }
}

// Sort key of entry e: its row, then (hub rows of the sliced layout) its group.
// `visit` (may be null): the keys are laid out in that order of the entries, key[v] = key of
// entry visit[v]; jj is in that order already.
template <typename KeyT>
__global__ void keys_k(const uint32_t *__restrict__ ii, const uint32_t *__restrict__ jj,
                       uint64_t nnz, bool slices, const uint8_t *__restrict__ hubflag,
                       const uint8_t *__restrict__ cls, const uint32_t *__restrict__ visit,
                       KeyT *key)
{
    GRID_STRIDE(v, nnz)
    {
        const uint32_t r = ii[visit ? visit[v] : v];
        if (!slices) {
            key[v] = (KeyT)r;
        } else {
            const uint32_t g = hubflag[r] ? hub_group(r, cls[jj[v]]) : 0u;
            key[v] = (KeyT)(((KeyT)r << 4) | (KeyT)g);
        }
    }
}

// ---- entries that come in the order of their rows ------------------------------------
// Kernel order is then the caller's but for the entries of hub rows (sliced layout), which go by group inside their
// row, in a group in their order.  A wavefront takes kOrderChunk entries, 64 at a time, and lane g keeps the count of
// group g in the row at hand; what a row has in chunks before is in `tail` (its first chunk) and `head` (the others).
// Bound by the reads of ii, jj and the tables: 16.8 M entries, 10 M of them of hub rows, 185 us (the same by a
// sort on row and group, the counting of its runs and a gather of the columns: 650).
// A chunk adds up what its row has in all chunks before: rows of more than kOrderRow entries are left to the sort
// (plans with one row of 8 M among 24 M entries 4.40 -> 4.03 ms, 16 M of 32 M 6.76 -> 6.71, 32 M of 48 M 11.4 -> 12.4).
constexpr uint32_t kOrderChunk = 1024;
constexpr uint32_t kOrderRow = 1u << 24;
constexpr uint32_t kGroups = 9;
struct OrderOut {
    uint32_t *hubcnt, *head, *tail; // counting: of every hub row its groups; of every chunk its first and its last row's
    uint32_t *perm, *col; // placing
    Counters *C;
};
template <bool PLACE>
__global__ void order_sorted_k(const uint32_t *__restrict__ ii, const uint32_t *__restrict__ jj, uint64_t nnz,
                               const uint8_t *__restrict__ hubflag, const uint32_t *__restrict__ hubpos,
                               const uint32_t *__restrict__ rowptr, const uint8_t *__restrict__ cls, OrderOut out)
{
    constexpr int U = 4; // batches in flight
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t chunk = ((uint64_t)blockIdx.x * kTB + threadIdx.x) / 64, lo = chunk * kOrderChunk;
    const uint64_t hi = lo + kOrderChunk < nnz ? lo + kOrderChunk : nnz;
    bool moved = false;
    uint32_t cur = 0xFFFFFFFFu, mine = 0, start = 0, end = 0; // the hub row at hand: lane g's count or next position
    const uint32_t head_row = lo < nnz ? ii[lo] : 0u;
    auto row_ends = [&] {
        if (PLACE || cur == 0xFFFFFFFFu || lane >= kGroups)
            return;
        const uint64_t at = (uint64_t)hubpos[cur] * kGroups + lane;
        if (start >= lo && end <= hi)
            out.hubcnt[at] = mine;
        else if (mine)
            atomicAdd(out.hubcnt + at, mine);
        if (cur == head_row)
            out.head[chunk * kGroups + lane] = mine;
    };
    auto row_begins = [&](uint32_t row) {
        cur = row;
        start = rowptr[row];
        end = rowptr[row + 1];
        mine = 0;
        if (!PLACE)
            return;
        uint32_t before = 0; // in chunks before this one, 7 of them at a time
        if (start < lo) {
            const uint64_t c0 = start / kOrderChunk;
            const uint32_t g = lane % kGroups, q = lane / kGroups;
            if (q < 7)
                for (uint64_t c = c0 + q; c < chunk; c += 7)
                    before += (c == c0 ? out.tail : out.head)[c * kGroups + g];
            uint32_t sum = 0;
            for (uint32_t i = 0; i < 7; ++i)
                sum += __shfl(before, (int)(i * kGroups + g), 64);
            before = sum;
        }
        const uint32_t n = lane < kGroups ? out.hubcnt[(uint64_t)hubpos[row] * kGroups + lane] : 0u;
        uint32_t upto = n;
        for (uint32_t d = 1; d < 16; d <<= 1) {
            const uint32_t o = __shfl_up(upto, d, 64);
            upto += lane >= d ? o : 0u;
        }
        mine = start + upto - n + before;
    };
    for (uint64_t e0 = lo; e0 < hi; e0 += 64 * U) {
        uint32_t r[U], c[U], g[U];
        bool on[U], hub[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t e = e0 + u * 64 + lane;
            on[u] = e < hi;
            r[u] = ii[on[u] ? e : lo];
            c[u] = jj[on[u] ? e : lo];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            hub[u] = on[u] && hubflag[r[u]];
            g[u] = hub_group(r[u], cls[c[u]]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t e = (uint32_t)(e0 + u * 64 + lane);
            uint32_t at = e;
            unsigned long long left = __ballot(hub[u]);
            if (left) {
                unsigned long long of_lane = 0, own = 0; // lanes of group `lane`, and of this entry's
                for (uint32_t k = 0; k < kGroups; ++k) {
                    const unsigned long long m = __ballot(hub[u] && g[u] == k);
                    of_lane = lane == k ? m : of_lane;
                    own = g[u] == k ? m : own;
                }
                while (left) {
                    const uint32_t row = (uint32_t)__shfl((int)r[u], __ffsll((long long)left) - 1, 64);
                    const unsigned long long here = __ballot(hub[u] && r[u] == row);
                    if (row != cur) {
                        row_ends();
                        row_begins(row);
                    }
                    if (PLACE) {
                        const uint32_t first = (uint32_t)__shfl((int)mine, (int)g[u], 64);
                        if (here >> lane & 1)
                            at = first + (uint32_t)__popcll(own & here & ((1ull << lane) - 1));
                    }
                    mine += (uint32_t)__popcll(of_lane & here);
                    left &= ~here;
                }
            }
            if (PLACE && on[u]) {
                out.perm[at] = e;
                out.col[at] = c[u];
                moved |= at != e;
            }
        }
    }
    row_ends();
    if (!PLACE) {
        if (cur != 0xFFFFFFFFu && lane < kGroups)
            out.tail[chunk * kGroups + lane] = mine;
        return;
    }
    if (__syncthreads_or(moved) && threadIdx.x == 0 &&
        !__hip_atomic_load(&out.C->not_identity, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicOr(&out.C->not_identity, 1u);
}

// col[p] = jj[perm[p]]; flags an order that is not the identity (one atomic per workgroup, and
// none once the flag is seen to be up).
__global__ void gather_cols_k(const uint32_t *__restrict__ jj, const uint32_t *__restrict__ perm,
                              uint64_t nnz, uint32_t *col, Counters *C)
{
    bool moved = false;
    GRID_STRIDE(p, nnz)
    {
        const uint32_t e = perm[p];
        col[p] = jj[e];
        moved |= e != (uint32_t)p;
    }
    if (__syncthreads_or(moved) && threadIdx.x == 0 &&
        !__hip_atomic_load(&C->not_identity, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicOr(&C->not_identity, 1u);
}

__device__ __forceinline__ uint32_t parts_of(uint32_t len, uint32_t seg_max)
{
    return len == 0 ? 0u : (len + seg_max - 1) / seg_max;
}

// Pieces per row; rows cut into several pieces also count as a split row and
// take one partial-sum slot per piece.
__global__ void count_pieces_k(const uint32_t *__restrict__ rowcnt, uint32_t nrows,
                               uint32_t seg_max, bool slices,
                               const uint8_t *__restrict__ hubflag,
                               const uint32_t *__restrict__ hubpos,
                               const uint32_t *__restrict__ hubcnt, uint32_t *npieces,
                               uint32_t *issplit, uint32_t *nslot)
{
    GRID_STRIDE(r, (uint64_t)nrows + 1)
    {
        uint32_t np = 0;
        if (r < nrows) {
            if (slices && hubflag[r]) {
                for (uint32_t k = 0; k < 9; ++k)
                    np += parts_of(hubcnt[(size_t)hubpos[r] * 9 + k], seg_max);
            } else {
                np = parts_of(rowcnt[r], seg_max);
            }
        }
        npieces[r] = np;
        issplit[r] = np > 1;
        nslot[r] = np > 1 ? np : 0u;
    }
}

// Writes the pieces of every row, in row order: balanced parts of at most
// seg_max entries per range (a non-hub row is one range, a hub row one per group).
__global__ void emit_pieces_k(const uint32_t *__restrict__ rowptr, uint32_t nrows,
                              uint32_t seg_max, bool slices,
                              const uint8_t *__restrict__ hubflag,
                              const uint32_t *__restrict__ hubpos,
                              const uint32_t *__restrict__ hubcnt,
                              const uint32_t *__restrict__ piece_off,
                              const uint32_t *__restrict__ split_off,
                              const uint32_t *__restrict__ slot_off, Seg *pseg, uint8_t *pqueue,
                              SplitRow *splits)
{
    GRID_STRIDE(r, nrows)
    {
        const uint32_t np = piece_off[r + 1] - piece_off[r];
        if (np == 0)
            continue;
        const uint32_t s = rowptr[r], len = rowptr[r + 1] - s;
        const bool hub = slices && hubflag[r];
        uint32_t at = piece_off[r];
        uint32_t slot = np > 1 ? slot_off[r] : kWholeRow;
        if (np > 1)
            splits[split_off[r]] = SplitRow{(uint32_t)r, slot_off[r], np, 0u};
        uint32_t start = s;
        const uint32_t ngroups = hub ? 9u : 1u;
        for (uint32_t k = 0; k < ngroups; ++k) {
            const uint32_t n = hub ? hubcnt[(size_t)hubpos[r] * 9 + k] : len;
            if (n == 0)
                continue;
            const uint8_t queue = (hub && k < 8) ? (uint8_t)k : kAnyQueue;
            const uint32_t parts = (n + seg_max - 1) / seg_max;
            const uint32_t base = n / parts, rem = n % parts;
            for (uint32_t q = 0; q < parts; ++q) {
                const uint32_t l = base + (q < rem ? 1u : 0u);
                pseg[at] = Seg{(uint32_t)r, start, l, slot};
                pqueue[at] = queue;
                ++at;
                start += l;
                if (np > 1)
                    ++slot;
            }
        }
    }
}

// Unsliced layout: key for "longest first", and the number of long pieces.
__global__ void len_keys_k(const Seg *__restrict__ pseg, uint64_t n, uint32_t seg_max,
                           uint32_t *key, Counters *C)
{
    uint32_t nl = 0;
    GRID_STRIDE(i, n)
    {
        const uint32_t l = pseg[i].len;
        key[i] = seg_max - l;
        nl += l >= kLongSegment;
    }
    nl = block_sum(nl);
    if (threadIdx.x == 0 && nl)
        atomicAdd(&C->nlong, nl);
}

__global__ void gather_segs_k(const Seg *__restrict__ pseg, const uint32_t *__restrict__ idx,
                              uint64_t n, Seg *out)
{
    GRID_STRIDE(i, n) out[i] = pseg[idx[i]];
}

// Sliced layout, step 1: the slice a free piece (any queue) prefers, which is the one most of its
// sliced entries belong to; kNoPref without any.  A group of 16 lanes per piece, four columns of a
// lane in flight: a thread per piece waited for two dependent loads per entry (R-MAT 20, 700 k
// pieces: 709 us, so 113).
constexpr uint32_t kPrefLanes = 16;
__global__ void pref_k(const Seg *__restrict__ pseg, const uint8_t *__restrict__ pqueue, uint64_t n,
                       const uint32_t *__restrict__ col, const uint8_t *__restrict__ cls,
                       uint8_t *pref)
{
    const uint32_t sub = threadIdx.x % kPrefLanes;
    GRID_STRIDE(t, n * kPrefLanes) // a group's lanes go round together
    {
        const uint64_t i = t / kPrefLanes;
        uint8_t p = kNoPref;
        if (pqueue[i] == kAnyQueue) {
            const Seg g = pseg[i];
            uint32_t cnt[kSlices] = {0};
            for (uint32_t q = sub; q < g.len; q += 4 * kPrefLanes) {
                uint32_t c[4];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u)
                    c[u] = col[g.start + (q + u * kPrefLanes < g.len ? q + u * kPrefLanes : q)];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) {
                    const uint32_t s = q + u * kPrefLanes < g.len ? cls[c[u]] : 255u;
#pragma unroll
                    for (uint32_t k = 0; k < kSlices; ++k)
                        cnt[k] += s == k;
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < kSlices; ++k)
#pragma unroll
                for (int s = kPrefLanes / 2; s >= 1; s >>= 1)
                    cnt[k] += __shfl_xor(cnt[k], s, kPrefLanes);
            // ties go to the first slice from a start that the row's hash picks
            const uint32_t first = rep_slice(g.row);
            uint32_t best = first, most = 0;
#pragma unroll
            for (uint32_t k = 0; k < kSlices; ++k)
                most = k == first ? cnt[k] : most;
            for (uint32_t k = 1; k < kSlices; ++k) {
                const uint32_t q = (first + k) % kSlices;
                uint32_t c = 0;
#pragma unroll
                for (uint32_t j = 0; j < kSlices; ++j)
                    c = j == q ? cnt[j] : c;
                if (c > most) {
                    most = c;
                    best = q;
                }
            }
            if (most)
                p = (uint8_t)best;
        }
        if (sub == 0)
            pref[i] = p;
    }
}

// Step 1b: which pieces are free, the work already bound to each queue, the free work, and the free
// work that prefers each slice.
__global__ void any_flags_k(const Seg *__restrict__ pseg, const uint8_t *__restrict__ pqueue,
                            const uint8_t *__restrict__ pref, uint64_t n, uint32_t *anyflag, Counters *C)
{
    unsigned long long w[2 * kSlices + 1] = {0}; // [8] = free work
    GRID_STRIDE(i, (uint64_t)n + 1)
    {
        if (i == n) {
            anyflag[i] = 0;
            continue;
        }
        const uint8_t q = pqueue[i], p = pref[i];
        const unsigned long long wi = (unsigned long long)pseg[i].len + kSegCost;
        anyflag[i] = q == kAnyQueue;
#pragma unroll
        for (uint32_t k = 0; k < kSlices; ++k) {
            w[k] += q == k ? wi : 0ull;
            w[kSlices + 1 + k] += q == kAnyQueue && p == k ? wi : 0ull;
        }
        w[kSlices] += q == kAnyQueue ? wi : 0ull;
    }
#pragma unroll
    for (uint32_t k = 0; k < 2 * kSlices + 1; ++k) {
        const unsigned long long t = block_sum(w[k]);
        if (threadIdx.x == 0 && t)
            atomicAdd(k < kSlices ? &C->load[k] : k == kSlices ? &C->any_load : &C->pref_load[k - kSlices - 1], t);
    }
}

// Step 2: the free pieces, compacted in piece order, with their length keys.
__global__ void compact_any_k(const Seg *__restrict__ pseg, const uint32_t *__restrict__ anyflag,
                              const uint32_t *__restrict__ anypos, uint64_t n, uint32_t seg_max,
                              uint32_t *any_idx, uint32_t *any_key)
{
    GRID_STRIDE(i, n)
    if (anyflag[i]) {
        any_idx[anypos[i]] = (uint32_t)i;
        any_key[anypos[i]] = seg_max - pseg[i].len;
    }
}


// Step 3: every piece gets its queue.  The combined list is [bound pieces in piece
// order | free pieces longest first]; its key is (queue, seg_max - len).
__global__ void combine_k(const Seg *__restrict__ pseg, const uint8_t *__restrict__ pqueue,
                          const uint32_t *__restrict__ anyflag,
                          const uint32_t *__restrict__ anypos,
                          const uint32_t *__restrict__ any_sorted,
                          const uint8_t *__restrict__ pref, uint64_t npieces, uint64_t nany,
                          uint32_t seg_max, DealPlan deal, uint32_t *comb_idx, uint32_t *comb_key,
                          Counters *C)
{
    const uint64_t nbound = npieces - nany;
    uint32_t cnt[kSlices] = {0}, lng[kSlices] = {0};
    GRID_STRIDE(t, npieces + nany)
    {
        uint32_t piece, q;
        uint64_t at;
        if (t < npieces) { // a bound piece, at its rank among the bound ones
            if (anyflag[t])
                continue;
            piece = (uint32_t)t;
            q = pqueue[t];
            at = t - anypos[t];
        } else { // the free piece of rank j
            const uint64_t j = t - npieces;
            piece = any_sorted[j];
            q = deal_queue_pref((uint32_t)j, pref[piece], deal);
            at = nbound + j;
        }
        const uint32_t l = pseg[piece].len;
        comb_idx[at] = piece;
        comb_key[at] = q * (seg_max + 1) + (seg_max - l);
#pragma unroll
        for (uint32_t k = 0; k < kSlices; ++k) {
            cnt[k] += q == k;
            lng[k] += q == k && l >= kLongSegment;
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < kSlices; ++k) {
        const uint32_t c = block_sum(cnt[k]), g = block_sum(lng[k]);
        if (threadIdx.x == 0) {
            if (c)
                atomicAdd(&C->qcount[k], c);
            if (g)
                atomicAdd(&C->qlong[k], g);
        }
    }
}

struct QStart {
    uint32_t v[kSlices];
};

// Step 4: piece of rank i in queue q goes to chunk i / 64 of that queue, which is
// global chunk (i / 64) * 8 + q.
__global__ void scatter_segs_k(const Seg *__restrict__ pseg, const uint32_t *__restrict__ idx,
                               const uint32_t *__restrict__ key, uint64_t n, uint32_t seg_max,
                               QStart qstart, Seg *out)
{
    GRID_STRIDE(s, n)
    {
        const uint32_t q = key[s] / (seg_max + 1);
        const uint64_t i = s - qstart.v[q];
        out[((i / kChunk) * kSlices + q) * kChunk + i % kChunk] = pseg[idx[s]];
    }
}

// ---- localizeIndices / ReMapIndices on the device -----------------------------
// head[i] = 1 where a run of equal sorted keys starts (i == n: 0, the scan's total slot)
__global__ void heads_k(const uint32_t *__restrict__ key, uint64_t n, uint32_t *head)
{
    GRID_STRIDE(i, n + 1) head[i] = (i < n && (i == 0 || key[i] != key[i - 1])) ? 1u : 0u;
}

// For every run: the position at which its value first appears in the caller's
// array (the sort is stable, so the head of the run holds it) and the value.
__global__ void run_firsts_k(const uint32_t *__restrict__ key, const uint32_t *__restrict__ pos,
                             const uint32_t *__restrict__ head,
                             const uint32_t *__restrict__ run_of, uint64_t n, uint32_t *first_pos,
                             uint32_t *run_key)
{
    GRID_STRIDE(i, n)
    if (head[i]) {
        first_pos[run_of[i]] = pos[i];
        run_key[run_of[i]] = key[i];
    }
}

// Runs in order of first appearance: the r-th gets local id r.
__global__ void run_ranks_k(const uint32_t *__restrict__ run_order,
                            const uint32_t *__restrict__ run_key, uint64_t nruns,
                            uint32_t *rank_of, uint32_t *ltg)
{
    GRID_STRIDE(r, nruns)
    {
        rank_of[run_order[r]] = (uint32_t)r;
        ltg[r] = run_key[run_order[r]];
    }
}

__global__ void write_local_k(const uint32_t *__restrict__ pos, const uint32_t *__restrict__ head,
                              const uint32_t *__restrict__ run_of,
                              const uint32_t *__restrict__ rank_of, uint64_t n, uint32_t *idx)
{
    // run_of[] is the exclusive scan of head[]: inside a run it already counts the head
    GRID_STRIDE(i, n) idx[pos[i]] = rank_of[run_of[i] + head[i] - 1];
}

__global__ void remap_check_k(const uint32_t *__restrict__ idx, uint64_t n, uint32_t map_len,
                              Counters *C)
{
    GRID_STRIDE(e, n)
    if (idx[e] >= map_len)
        atomicMin(&C->first_bad, (uint32_t)e);
}

// Changes nothing when the check found an index outside the map.
__global__ void remap_apply_k(uint32_t *idx, uint64_t n, const uint32_t *__restrict__ map,
                              const Counters *__restrict__ C)
{
    if (C->first_bad != 0xFFFFFFFFu)
        return;
    GRID_STRIDE(e, n) idx[e] = map[idx[e]];
}

#define HIP_OK(expr)                                                                              \
    do {                                                                                          \
        const hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess) {                                                                   \
            err = std::string("device plan: ") + #expr + ": " + hipGetErrorString(e_);            \
            return e_ == hipErrorOutOfMemory ? SPC3D_ERR_ALLOC : SPC3D_ERR_HIP;                   \
        }                                                                                         \
    } while (0)

// Scratch for the device-wide primitives, grown on demand.
struct Temp {
    Arena &arena;
    unsigned char *p = nullptr;
    size_t cap = 0;
    explicit Temp(Arena &a) : arena(a) {}
    hipError_t need(size_t bytes)
    {
        bytes = bytes < 256 ? 256 : bytes; // never null: a null pointer asks for the size again
        if (bytes <= cap)
            return hipSuccess;
        const hipError_t e = arena.take(reinterpret_cast<void **>(&p), bytes);
        cap = e == hipSuccess ? bytes : 0;
        return e;
    }
};

template <typename T>
int exclusive_sum(Temp &tmp, const T *in, uint32_t *out, size_t n, const DevStream &st, std::string &err)
{
    size_t bytes = 0;
    HIP_OK(rocprim::exclusive_scan(nullptr, bytes, in, out, 0u, n, rocprim::plus<uint32_t>(), st));
    HIP_OK(tmp.need(bytes));
    HIP_OK(rocprim::exclusive_scan(tmp.p, bytes, in, out, 0u, n, rocprim::plus<uint32_t>(), st));
    return SPC3D_OK;
}

// By digits from 64 k items on: below a million the primitive's own choice is a merge sort, whose two
// kernels per doubling cost more (1 M pairs: 260 us).
using SortConfig =
    rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config, rocprim::default_config, 1u << 16>;

// Stable ascending sort of (key, value) pairs on key bits [0, bits).
template <typename KeyT>
int sort_pairs(Temp &tmp, const KeyT *kin, KeyT *kout, const uint32_t *vin, uint32_t *vout,
               uint32_t n, int bits, bool descending, const DevStream &st, std::string &err)
{
    size_t bytes = 0;
    if (descending) {
        HIP_OK(rocprim::radix_sort_pairs_desc<SortConfig>(nullptr, bytes, kin, kout, vin, vout, (size_t)n, 0u,
                                              (unsigned)bits, st));
        HIP_OK(tmp.need(bytes));
        HIP_OK(rocprim::radix_sort_pairs_desc<SortConfig>(tmp.p, bytes, kin, kout, vin, vout, (size_t)n, 0u,
                                              (unsigned)bits, st));
    } else {
        HIP_OK(rocprim::radix_sort_pairs<SortConfig>(nullptr, bytes, kin, kout, vin, vout, (size_t)n, 0u,
                                         (unsigned)bits, st));
        HIP_OK(tmp.need(bytes));
        HIP_OK(rocprim::radix_sort_pairs<SortConfig>(tmp.p, bytes, kin, kout, vin, vout, (size_t)n, 0u,
                                         (unsigned)bits, st));
    }
    return SPC3D_OK;
}

#define LAUNCH(kernel, n, ...)                                                                    \
    hipLaunchKernelGGL(kernel, dim3(grid_for(n)), dim3(kTB), 0, st, __VA_ARGS__)
#define LAUNCH_SMALL(kernel, n, ...)                                                              \
    hipLaunchKernelGGL(kernel, dim3(small_grid_for(n)), dim3(kTB), 0, st, __VA_ARGS__)

#define LAUNCH_FEW(kernel, n, ...)                                                                \
    hipLaunchKernelGGL(kernel, dim3(few_grid_for(n)), dim3(kTB), 0, st, __VA_ARGS__)

#define TRY(expr)                                                                                 \
    do {                                                                                          \
        const int rc_ = (expr);                                                                   \
        if (rc_ != SPC3D_OK)                                                                      \
            return rc_;                                                                           \
    } while (0)

// cnt[id] = how often id < nbins comes among n ids of an arbitrary order.  A device-wide atomic per entry is
// served at the memory side, 1.5 ms for 16.8 M; sorting the ids and finding the runs takes 320 us; what is done, one
// digit of that sort at most (to 4 M bins) and counters in LDS, 190.  `scratch` is for n ids.
int count_ids(Temp &tmp, Arena &arena, const uint32_t *ids, uint32_t n, uint32_t nbins, uint32_t *scratch,
              uint32_t *cnt, const DevStream &st, std::string &err)
{
    const uint32_t bits = (uint32_t)bits_for(nbins ? nbins - 1 : 0);
    const CountSizes sizes = count_sizes(n, nbins);
    const uint32_t low = sizes.low, nbuckets = sizes.nbuckets, part = sizes.part, most = sizes.most;
    if (low < bits) {
        size_t bytes = 0;
        HIP_OK(rocprim::radix_sort_keys<SortConfig>(nullptr, bytes, ids, scratch, (size_t)n, low, bits, st));
        HIP_OK(tmp.need(bytes));
        HIP_OK(rocprim::radix_sort_keys<SortConfig>(tmp.p, bytes, ids, scratch, (size_t)n, low, bits, st));
        ids = scratch;
    }
    SBuf<uint32_t> start, parts, first_part, counts;
    HIP_OK(start.alloc(arena, (size_t)nbuckets + 1));
    HIP_OK(parts.alloc(arena, (size_t)nbuckets + 1));
    HIP_OK(first_part.alloc(arena, (size_t)nbuckets + 1));
    HIP_OK(counts.alloc(arena, (size_t)most << low));
    hipLaunchKernelGGL(bucket_parts_k, dim3(nbuckets / (kTB / 64) + 1), dim3(kTB), 0, st, ids, n, low, nbuckets, part,
                       start.p, parts.p);
    TRY(exclusive_sum(tmp, parts.p, first_part.p, (size_t)nbuckets + 1, st, err));
    hipLaunchKernelGGL(bucket_count_k, dim3(most), dim3(kCountTB), 0, st, ids, start.p, first_part.p, low, nbuckets,
                       part, counts.p);
    LAUNCH(bucket_sum_k, nbins, counts.p, first_part.p, low, (uint64_t)nbins, cnt);
    return SPC3D_OK;
}

struct Fetch { // bytes from dev to host
    void *host;
    const void *dev;
    size_t bytes;
};
// Waits for what is queued on the stream and brings the given words down, through pinned memory
// (into pageable memory each wait takes 15 us more, and a plan has seven or more).
int fetch_all(const DevStream &st, std::initializer_list<Fetch> list, std::string &err)
{
    HIP_OK(hipGetLastError());
    size_t need = 0;
    for (const Fetch &f : list)
        need += (f.bytes + 15) / 16 * 16;
    void *words = need <= DevPool::kWords ? st.pool->get_words() : nullptr;
    hipError_t e = hipSuccess;
    char *at = static_cast<char *>(words);
    for (const Fetch &f : list) {
        if (e == hipSuccess)
            e = hipMemcpyAsync(words ? at : f.host, f.dev, f.bytes, hipMemcpyDeviceToHost, st);
        at += words ? (f.bytes + 15) / 16 * 16 : 0;
    }
    const hipError_t done = hipStreamSynchronize(st); // also before the words are given back
    e = e == hipSuccess ? done : e;
    at = static_cast<char *>(words);
    if (words && e == hipSuccess)
        for (const Fetch &f : list) {
            std::memcpy(f.host, at, f.bytes);
            at += (f.bytes + 15) / 16 * 16;
        }
    st.pool->put_words(words);
    HIP_OK(e);
    return SPC3D_OK;
}
int fetch(const DevStream &st, void *host, const void *dev, size_t bytes, std::string &err)
{
    return fetch_all(st, {{host, dev, bytes}}, err);
}

// Sorts the entries into kernel order: perm (kernel position -> caller's
// position) and col.  KeyT is wide enough for (row << 4 | group).  hubcnt (sliced layout): see
// hubcount_k.
// visit (may be null): the entries in ascending column order (stable), so that every row ends
// up ordered by column; col then holds the columns in that order.
template <typename KeyT>
int order_entries(Arena &arena, Temp &tmp, const DevStream &st, uint64_t nnz, int key_bits, bool slices,
                  const uint32_t *visit, const uint32_t *d_ii, const uint32_t *d_jj,
                  const uint8_t *hubflag, const uint32_t *hubpos, uint32_t *hubcnt,
                  const uint8_t *cls, uint32_t *perm, uint32_t *col, Counters *C, std::string &err)
{
    SBuf<KeyT> key, key_out;
    SBuf<uint32_t> ident;
    HIP_OK(key.alloc(arena, nnz));
    HIP_OK(key_out.alloc(arena, nnz));
    if (!visit) {
        HIP_OK(ident.alloc(arena, nnz));
        LAUNCH(iota_k, nnz, ident.p, nnz);
    }
    LAUNCH((keys_k<KeyT>), nnz, d_ii, visit ? col : d_jj, nnz, slices, hubflag, cls, visit, key.p);
    TRY(sort_pairs<KeyT>(tmp, key.p, key_out.p, visit ? visit : ident.p, perm, (uint32_t)nnz, key_bits,
                         false, st, err));
    if (slices)
        LAUNCH((hubcount_k<KeyT>), nnz, key_out.p, nnz, hubflag, hubpos, hubcnt);
    LAUNCH(gather_cols_k, nnz, d_jj, perm, nnz, col, C);
    HIP_OK(hipGetLastError());
    return SPC3D_OK;
}

// The same for entries that come in the order of their rows (hubcnt zeroed; not sliced: the caller's order).
int order_sorted_entries(Arena &arena, const DevStream &st, uint64_t nnz, bool slices, const uint32_t *d_ii,
                         const uint32_t *d_jj, const uint8_t *hubflag, const uint32_t *hubpos, uint32_t *hubcnt,
                         const uint32_t *rowptr, const uint8_t *cls, uint32_t *perm, uint32_t *col, Counters *C,
                         std::string &err)
{
    if (!slices) {
        LAUNCH(iota_k, nnz, perm, nnz);
        HIP_OK(hipMemcpyAsync(col, d_jj, (size_t)nnz * sizeof(uint32_t), hipMemcpyDeviceToDevice, st));
        return SPC3D_OK;
    }
    const uint64_t nchunks = (nnz + kOrderChunk - 1) / kOrderChunk;
    SBuf<uint32_t> head, tail;
    HIP_OK(head.alloc(arena, nchunks * kGroups));
    HIP_OK(tail.alloc(arena, nchunks * kGroups));
    const OrderOut out = {hubcnt, head.p, tail.p, perm, col, C};
    const dim3 grid((uint32_t)((nchunks + kTB / 64 - 1) / (kTB / 64)));
    hipLaunchKernelGGL(order_sorted_k<false>, grid, dim3(kTB), 0, st, d_ii, d_jj, nnz, hubflag, hubpos, rowptr, cls, out);
    hipLaunchKernelGGL(order_sorted_k<true>, grid, dim3(kTB), 0, st, d_ii, d_jj, nnz, hubflag, hubpos, rowptr, cls, out);
    HIP_OK(hipGetLastError());
    return SPC3D_OK;
}

// ---- column blocks ---------------------------------------------------------------
__global__ void block_keys_k(const uint32_t *__restrict__ jj, uint64_t nnz, uint32_t block_cols,
                             uint32_t *key)
{
    GRID_STRIDE(e, nnz) key[e] = jj[e] / block_cols;
}
__global__ void gather_u32_k(const uint32_t *__restrict__ in, const uint32_t *__restrict__ idx,
                             uint64_t n, uint32_t *out)
{
    GRID_STRIDE(e, n) out[e] = in[idx[e]];
}
// first[b] = position of the first entry of block b in the sorted keys (first[nblocks] = n)
__global__ void block_firsts_k(const uint32_t *__restrict__ sorted, uint64_t n, uint32_t nblocks,
                               uint32_t *first)
{
    GRID_STRIDE(i, n + 1)
    {
        const uint32_t lo = i == 0 ? 0u : sorted[i - 1] + 1;
        const uint32_t hi = i == n ? nblocks : sorted[i];
        for (uint32_t b = lo; b <= hi && b <= nblocks; ++b)
            first[b] = (uint32_t)i;
    }
}
// perm[q] = order[off + (perm ? perm[q] : q)]
__global__ void compose_perm_k(const uint32_t *__restrict__ order, const uint32_t *__restrict__ perm,
                               uint64_t n, uint32_t *out)
{
    GRID_STRIDE(q, n) out[q] = order[perm ? perm[q] : (uint32_t)q];
}
// out[perm[q]] = vals[q]
__global__ void scatter_u32_k(const uint32_t *__restrict__ perm, const uint32_t *__restrict__ vals,
                              uint64_t n, uint32_t *out)
{
    GRID_STRIDE(q, n) out[perm[q]] = vals[q];
}
// key[q] = rows[perm ? perm[q] : q] / rows_per_tile
__global__ void tile_keys_k(const uint32_t *__restrict__ rows, const uint32_t *__restrict__ perm,
                            uint64_t n, uint32_t rows_per_tile, uint32_t *key)
{
    GRID_STRIDE(q, n) key[q] = rows[perm ? perm[q] : (uint32_t)q] / rows_per_tile;
}
// rank[sorted[i]] = i
__global__ void ranks_k(const uint32_t *__restrict__ sorted, uint64_t n, uint32_t *rank)
{
    GRID_STRIDE(i, n) rank[sorted[i]] = (uint32_t)i;
}

} // namespace

int build_device_plan(const DevStream &st, uint32_t nrows, uint32_t ncols, uint64_t nnz,
                      const uint32_t *d_ii, const uint32_t *d_jj, const PlanOpts &opts,
                      HostPlan &meta, DevPlanArrays &out, std::string &err)
{
    if (nnz >= (1ull << 32)) {
        err = "nnz >= 2^32 is not supported";
        return SPC3D_ERR_TOO_LARGE;
    }
    if (nnz > 0 && (d_ii == nullptr || d_jj == nullptr)) {
        err = "ii/jj is NULL with nnz > 0";
        return SPC3D_ERR_INVALID_ARG;
    }
    const uint32_t hub_min = opts.hub_min ? opts.hub_min : kDefaultHubMin;
    const bool want_slices = opts.xcd_slices == 0 || opts.xcd_slices == kSlices;

    HostPlan P;
    P.nrows = nrows;
    P.ncols = ncols;
    P.nnz = nnz;
    out = DevPlanArrays{};
    if (nnz == 0) {
        P.seg_max = clamp_seg_max(
            opts.seg_max ? opts.seg_max : default_seg_max(nnz, opts.row_bytes, nrows, 0, 0), nnz);
        meta = std::move(P);
        return SPC3D_OK;
    }

    Arena arena(st);
    Temp tmp(arena);
    SBuf<Counters> dC;
    Counters hC;
    HIP_OK(arena.reserve(sizeof(Counters) + 256)); // (how much more is known when the entries are checked)
    HIP_OK(dC.alloc(arena, 1));
    HIP_OK(hipMemsetAsync(dC.p, 0, sizeof(Counters), st));
    HIP_OK(hipMemsetAsync(&dC.p->first_bad, 0xFF, sizeof(uint32_t), st));

    // ---- histograms, validation ------------------------------------------------
    LAUNCH_SMALL(check_k, nnz, d_ii, d_jj, nnz, nrows, ncols, dC.p);
    TRY(fetch(st, &hC, dC.p, sizeof hC, err));
    if (hC.first_bad != 0xFFFFFFFFu) {
        uint32_t r = 0, c = 0;
        TRY(fetch(st, &r, d_ii + hC.first_bad, sizeof r, err));
        TRY(fetch(st, &c, d_jj + hC.first_bad, sizeof c, err));
        char buf[160];
        std::snprintf(buf, sizeof buf, "entry %llu = (%u, %u) is outside the %u x %u pattern",
                      (unsigned long long)hC.first_bad, r, c, nrows, ncols);
        err = buf;
        return SPC3D_ERR_BAD_INDEX;
    }
    const bool rows_unsorted = hC.rows_unsorted != 0;
    P.cols_sorted = hC.cols_unsorted == 0;
    P.rows_sorted = !rows_unsorted;
    P.row_runs = hC.row_changes + 1; // (nnz > 0)
    const bool by_column = rows_unsorted && !opts.keep_entry_order;
    const int col_bits = bits_for(ncols ? ncols - 1 : 0);
    P.by_column_in_rows = by_column;
    // Rows that come in runs are counted run by run (hist_sorted_k), which eight per run already pay for.
    const bool count_rows = rows_unsorted && (uint64_t)hC.row_changes * 8 > nnz;
    const CountSizes of_rows = count_sizes((uint32_t)nnz, nrows), of_cols = count_sizes((uint32_t)nnz, ncols);
    const bool sort_ids = by_column || of_cols.nbuckets > 1 || (count_rows && of_rows.nbuckets > 1);
    // One block for what is known to be needed: seven arrays of words and two of bytes per row, four and a byte per
    // column, the scratch of the columns' sort; per entry, where rows are sorted, the ids and the scratch of a sort of
    // theirs, with the counters of the ids, elsewhere two keys and two orders (the scratch of their sorts comes on top).
    {
        const size_t key_bytes = bits_for(nrows ? nrows - 1 : 0) + 4 > 32 ? 8 : 4;
        const size_t per_entry = rows_unsorted ? 2 * key_bytes + 8 : (sort_ids ? 8 : 0);
        const size_t counters = rows_unsorted ? 0 : (size_t)of_cols.most << of_cols.low;
        HIP_OK(arena.reserve(((size_t)nrows + 1) * 35 + (size_t)ncols * 26 + counters * 4 + (size_t)nnz * per_entry +
                             (size_t)nnz / 2 + ((size_t)8 << 20)));
    }
    SBuf<uint32_t> rowcnt;
    DBuf<uint32_t> rowptr, coldeg;
    HIP_OK(rowcnt.alloc(arena, (size_t)nrows + 1));
    HIP_OK(rowptr.alloc(st, (size_t)nrows + 1));
    HIP_OK(coldeg.alloc(st, ncols));
    HIP_OK(hipMemsetAsync(rowcnt.p, 0, ((size_t)nrows + 1) * sizeof(uint32_t), st));
    HIP_OK(hipMemsetAsync(coldeg.p, 0, (size_t)ncols * sizeof(uint32_t), st));
    DBuf<uint32_t> perm, col;
    SBuf<uint32_t> visit;
    HIP_OK(perm.alloc(st, nnz));
    HIP_OK(col.alloc(st, nnz));
    {
        SBuf<uint32_t> sorted, start;
        if (sort_ids)
            HIP_OK(sorted.alloc(arena, nnz));
        if (count_rows) {
            TRY(count_ids(tmp, arena, d_ii, (uint32_t)nnz, nrows, sorted.p, rowcnt.p, st, err));
        } else {
            LAUNCH(hist_sorted_k, nnz, d_ii, nnz, rowcnt.p);
        }
        if (by_column) { // the visiting order of order_entries; its sorted columns in `col`
            HIP_OK(visit.alloc(arena, nnz));
            HIP_OK(start.alloc(arena, ncols));
            LAUNCH(iota_k, nnz, sorted.p, nnz);
            TRY(sort_pairs<uint32_t>(tmp, d_jj, col.p, sorted.p, visit.p, (uint32_t)nnz, col_bits,
                                     false, st, err));
            LAUNCH(run_bounds_k, nnz, col.p, nnz, ncols, start.p, coldeg.p);
            LAUNCH(run_lengths_k, ncols, start.p, (uint64_t)ncols, coldeg.p);
        } else {
            TRY(count_ids(tmp, arena, d_jj, (uint32_t)nnz, ncols, sorted.p, coldeg.p, st, err));
        }
    }
    LAUNCH_FEW(stats_k, nrows, rowcnt.p, (uint64_t)nrows, &dC.p->rows_touched, &dC.p->max_row,
                 &dC.p->row_sq);
    LAUNCH_FEW(stats_k, ncols, coldeg.p, (uint64_t)ncols, &dC.p->cols_touched, &dC.p->max_cdeg,
                 (unsigned long long *)nullptr);
    TRY(exclusive_sum(tmp, rowcnt.p, rowptr.p, (size_t)nrows + 1, st, err));
    TRY(fetch(st, &hC, dC.p, sizeof hC, err));
    P.rows_touched = hC.rows_touched;
    P.cols_touched = hC.cols_touched;
    P.max_row_nnz = hC.max_row;
    P.row_sq = hC.row_sq;
    const uint32_t seg_max = clamp_seg_max(
        opts.seg_max ? opts.seg_max
                     : default_seg_max(nnz, opts.row_bytes, nrows, hC.rows_touched, hC.max_row), nnz);
    P.seg_max = seg_max;
    P.seg_shortened = !opts.seg_max && seg_max < seg_max_by_entries(nnz, opts.row_bytes);
    const uint32_t ctouched = hC.cols_touched, maxcdeg = hC.max_cdeg;

    // ---- column classes (XCD slicing only) ---------------------------------------
    SBuf<uint8_t> cls;
    DBuf<uint32_t> hot;
    bool slices = false;
    if (want_slices && opts.hot_cols > 0 && ctouched > opts.hot_cols) {
        const uint32_t h1 = opts.hot_cols;
        const uint32_t hrep = std::max<uint32_t>(h1 / 6, 1);
        const uint64_t htot =
            std::min<uint64_t>((uint64_t)hrep + (uint64_t)(h1 - hrep) * kSlices, ctouched);
        // Columns by degree, highest first, ties in column order (a stable sort);
        // the untouched columns end up last.
        SBuf<uint32_t> colid, order, deg_sorted;
        HIP_OK(colid.alloc(arena, ncols));
        HIP_OK(order.alloc(arena, ncols));
        HIP_OK(deg_sorted.alloc(arena, ncols));
        LAUNCH(iota_k, ncols, colid.p, (uint64_t)ncols);
        TRY(sort_pairs<uint32_t>(tmp, coldeg.p, deg_sorted.p, colid.p, order.p, ncols,
                                 bits_for(maxcdeg), true, st, err));
        LAUNCH_SMALL(sum_first_k, htot, deg_sorted.p, htot, &dC.p->covered);
        const bool hot_form = !opts.one_call && ncols <= kHotRow && hot_rows_pay(nnz, opts.hot_row_bytes);
        const uint32_t nhot = (uint32_t)std::min<uint64_t>(kHotRows, htot);
        if (hot_form)
            hipLaunchKernelGGL(hot_weight_k, dim3(1), dim3(kTB), 0, st, order.p, deg_sorted.p, nhot,
                               dC.p->hot_weight);
        TRY(fetch(st, &hC, dC.p, sizeof hC, err));
        const uint64_t covered = hC.covered;
        const double coverage = (double)covered / (double)nnz;
        const double share = (double)htot / (double)ctouched;
        if (coverage >= 0.2 && coverage >= 2.0 * share) {
            slices = true;
            HIP_OK(cls.alloc(arena, ncols));
            LAUNCH(fill_k<uint8_t>, ncols, cls.p, (uint64_t)ncols, kClsCold);
            LAUNCH(classify_k, htot, order.p, htot, hrep, cls.p);
            P.hot_cols = (uint32_t)htot;
            P.hot_entries = covered;
            uint64_t weight[kHotClasses];
            for (uint32_t i = 0; i < kHotClasses; ++i)
                weight[i] = hC.hot_weight[i];
            if (hot_form && hot_rows_crowd(weight)) {
                HIP_OK(hot.alloc(st, nhot));
                HIP_OK(hipMemcpyAsync(hot.p, order.p, nhot * sizeof(uint32_t), hipMemcpyDeviceToDevice, st));
                out.nhot = nhot;
            }
        }
        HIP_OK(hipGetLastError());
    }

    // ---- hub rows: group counts ---------------------------------------------------
    SBuf<uint8_t> hubflag;
    SBuf<uint32_t> hubpos, hubcnt;
    uint32_t nh = 0;
    if (slices) {
        HIP_OK(hubflag.alloc(arena, (size_t)nrows + 1));
        HIP_OK(hubpos.alloc(arena, (size_t)nrows + 1));
        LAUNCH(hubflag_k, (uint64_t)nrows + 1, rowcnt.p, nrows, hub_min, hubflag.p);
        TRY(exclusive_sum(tmp, hubflag.p, hubpos.p, (size_t)nrows + 1, st, err));
        TRY(fetch(st, &nh, hubpos.p + nrows, sizeof nh, err));
        P.hub_rows = nh;
        HIP_OK(hubcnt.alloc(arena, (size_t)nh * 9 + 1));
        HIP_OK(hipMemsetAsync(hubcnt.p, 0, ((size_t)nh * 9 + 1) * sizeof(uint32_t), st));
    }

    // ---- stable sort into kernel order ------------------------------------------------
    {
        const int key_bits = bits_for(nrows ? nrows - 1 : 0) + (slices ? 4 : 0);
        if (!rows_unsorted && (!slices || P.max_row_nnz <= kOrderRow))
            TRY(order_sorted_entries(arena, st, nnz, slices, d_ii, d_jj, hubflag.p, hubpos.p, hubcnt.p, rowptr.p,
                                     cls.p, perm.p, col.p, dC.p, err));
        else if (key_bits <= 32)
            TRY(order_entries<uint32_t>(arena, tmp, st, nnz, key_bits, slices, visit.p, d_ii, d_jj,
                                        hubflag.p, hubpos.p, hubcnt.p, cls.p, perm.p, col.p, dC.p,
                                        err));
        else
            TRY(order_entries<unsigned long long>(arena, tmp, st, nnz, key_bits, slices, visit.p,
                                                  d_ii, d_jj, hubflag.p, hubpos.p, hubcnt.p, cls.p,
                                                  perm.p, col.p, dC.p, err));
    }

    // ---- segments --------------------------------------------------------------------
    SBuf<uint32_t> npieces, issplit, nslot, piece_off, split_off, slot_off;
    const size_t nr1 = (size_t)nrows + 1;
    HIP_OK(npieces.alloc(arena, nr1));
    HIP_OK(issplit.alloc(arena, nr1));
    HIP_OK(nslot.alloc(arena, nr1));
    HIP_OK(piece_off.alloc(arena, nr1));
    HIP_OK(split_off.alloc(arena, nr1));
    HIP_OK(slot_off.alloc(arena, nr1));
    LAUNCH(count_pieces_k, nr1, rowcnt.p, nrows, seg_max, slices, hubflag.p, hubpos.p, hubcnt.p,
           npieces.p, issplit.p, nslot.p);
    TRY(exclusive_sum(tmp, npieces.p, piece_off.p, (size_t)nrows + 1, st, err));
    TRY(exclusive_sum(tmp, issplit.p, split_off.p, (size_t)nrows + 1, st, err));
    TRY(exclusive_sum(tmp, nslot.p, slot_off.p, (size_t)nrows + 1, st, err));
    uint32_t totals[3] = {0, 0, 0};
    TRY(fetch_all(st,
                  {{&totals[0], piece_off.p + nrows, sizeof(uint32_t)},
                   {&totals[1], split_off.p + nrows, sizeof(uint32_t)},
                   {&totals[2], slot_off.p + nrows, sizeof(uint32_t)}},
                  err));
    const uint32_t np_total = totals[0], nsplit = totals[1];
    P.nslots = totals[2];
    P.nseg_real = np_total;

    // and one for everything sized by the number of pieces
    HIP_OK(arena.reserve((size_t)np_total * 64 + ((size_t)4 << 20)));
    SBuf<Seg> pseg;
    SBuf<uint8_t> pqueue;
    DBuf<SplitRow> splits;
    HIP_OK(pseg.alloc(arena, np_total));
    HIP_OK(pqueue.alloc(arena, np_total));
    HIP_OK(splits.alloc(st, nsplit));
    LAUNCH(emit_pieces_k, nrows, rowptr.p, nrows, seg_max, slices, hubflag.p, hubpos.p, hubcnt.p,
           piece_off.p, split_off.p, slot_off.p, pseg.p, pqueue.p, splits.p);

    // ---- order and deal --------------------------------------------------------------
    DBuf<Seg> segs;
    uint32_t nseg_padded = 0;
    const int len_bits = bits_for(seg_max);
    if (!slices) {
        SBuf<uint32_t> key, key_out, idx, idx_out;
        HIP_OK(key.alloc(arena, np_total));
        HIP_OK(key_out.alloc(arena, np_total));
        HIP_OK(idx.alloc(arena, np_total));
        HIP_OK(idx_out.alloc(arena, np_total));
        HIP_OK(segs.alloc(st, np_total));
        LAUNCH_SMALL(len_keys_k, np_total, pseg.p, (uint64_t)np_total, seg_max, key.p, dC.p);
        LAUNCH(iota_k, np_total, idx.p, (uint64_t)np_total);
        TRY(sort_pairs<uint32_t>(tmp, key.p, key_out.p, idx.p, idx_out.p, np_total, len_bits,
                                 false, st, err));
        LAUNCH(gather_segs_k, np_total, pseg.p, idx_out.p, (uint64_t)np_total, segs.p);
        TRY(fetch(st, &hC, dC.p, sizeof hC, err));
        P.nqueues = 1;
        nseg_padded = np_total;
        P.nseg_long = hC.nlong / kChunk * kChunk;
    } else {
        SBuf<uint32_t> anyflag, anypos;
        SBuf<uint8_t> pref;
        HIP_OK(anyflag.alloc(arena, (size_t)np_total + 1));
        HIP_OK(anypos.alloc(arena, (size_t)np_total + 1));
        HIP_OK(pref.alloc(arena, np_total));
        LAUNCH(pref_k, (uint64_t)np_total * kPrefLanes, pseg.p, pqueue.p, (uint64_t)np_total, col.p,
               cls.p, pref.p);
        LAUNCH_FEW(any_flags_k, (uint64_t)np_total + 1, pseg.p, pqueue.p, pref.p, (uint64_t)np_total,
                   anyflag.p, dC.p);
        TRY(exclusive_sum(tmp, anyflag.p, anypos.p, (size_t)np_total + 1, st, err));
        uint32_t nany = 0;
        TRY(fetch_all(st, {{&nany, anypos.p + np_total, sizeof nany}, {&hC, dC.p, sizeof hC}}, err));

        SBuf<uint32_t> any_idx, any_key, any_key_out, any_sorted;
        HIP_OK(any_idx.alloc(arena, nany));
        HIP_OK(any_key.alloc(arena, nany));
        HIP_OK(any_key_out.alloc(arena, nany));
        HIP_OK(any_sorted.alloc(arena, nany));
        if (nany) {
            LAUNCH(compact_any_k, np_total, pseg.p, anyflag.p, anypos.p, (uint64_t)np_total,
                   seg_max, any_idx.p, any_key.p);
            TRY(sort_pairs<uint32_t>(tmp, any_key.p, any_key_out.p, any_idx.p, any_sorted.p, nany,
                                     len_bits, false, st, err));
        }
        uint64_t load[kDealQueues], pref_load[kDealQueues];
        for (uint32_t q = 0; q < kDealQueues; ++q) {
            load[q] = hC.load[q];
            pref_load[q] = hC.pref_load[q];
        }
        DealPlan deal;
        deal_plan(load, pref_load, hC.any_load, opts.slice_affinity, deal);

        SBuf<uint32_t> comb_idx, comb_key, comb_idx_out, comb_key_out;
        HIP_OK(comb_idx.alloc(arena, np_total));
        HIP_OK(comb_key.alloc(arena, np_total));
        HIP_OK(comb_idx_out.alloc(arena, np_total));
        HIP_OK(comb_key_out.alloc(arena, np_total));
        LAUNCH_FEW(combine_k, (uint64_t)np_total + nany, pseg.p, pqueue.p, anyflag.p, anypos.p,
               any_sorted.p, pref.p, (uint64_t)np_total, (uint64_t)nany, seg_max, deal, comb_idx.p,
               comb_key.p, dC.p);
        const int comb_bits = bits_for((uint64_t)kSlices * ((uint64_t)seg_max + 1) - 1);
        TRY(sort_pairs<uint32_t>(tmp, comb_key.p, comb_key_out.p, comb_idx.p, comb_idx_out.p,
                                 np_total, comb_bits, false, st, err));
        TRY(fetch(st, &hC, dC.p, sizeof hC, err));
        QStart qs;
        uint32_t at = 0, nchunks = 0, rounds = 0xFFFFFFFFu;
        for (uint32_t q = 0; q < kSlices; ++q) {
            qs.v[q] = at;
            at += hC.qcount[q];
            nchunks = std::max(nchunks, (hC.qcount[q] + kChunk - 1) / kChunk);
            rounds = std::min(rounds, hC.qlong[q] / kChunk);
        }
        const uint64_t padded = (uint64_t)nchunks * kSlices * kChunk;
        if (padded >= (1ull << 32)) {
            err = "the padded segment list does not fit 32 bits";
            return SPC3D_ERR_TOO_LARGE;
        }
        nseg_padded = (uint32_t)padded;
        HIP_OK(segs.alloc(st, nseg_padded));
        LAUNCH(fill_k<Seg>, nseg_padded, segs.p, (uint64_t)nseg_padded, (Seg{0, 0, 0, kWholeRow}));
        LAUNCH(scatter_segs_k, np_total, pseg.p, comb_idx_out.p, comb_key_out.p,
               (uint64_t)np_total, seg_max, qs, segs.p);
        P.nqueues = kSlices;
        P.nseg_long = rounds * kSlices * kChunk;
    }
    HIP_OK(hipGetLastError());
    HIP_OK(hipStreamSynchronize(st));
    P.identity = hC.not_identity == 0;

    out.segs = segs.release();
    out.nseg_padded = nseg_padded;
    out.col = col.release();
    out.perm = P.identity ? nullptr : perm.release();
    out.splits = splits.release();
    out.nsplit = nsplit;
    out.hot_cols = hot.release();
    if (opts.keep_counts && slices) {
        out.rowptr = rowptr.release();
        out.coldeg = coldeg.release();
    }
    meta = std::move(P);
    return SPC3D_OK;
}

int encode_hot_device(const DevStream &st, const uint32_t *d_col, uint64_t n, const uint32_t *d_hot,
                      uint32_t nhot, uint32_t ncols, uint32_t *d_out, std::string &err)
{
    DBuf<uint16_t> rank;
    HIP_OK(rank.alloc(st, ncols));
    LAUNCH(fill_k<uint16_t>, ncols, rank.p, (uint64_t)ncols, (uint16_t)0xFFFFu);
    LAUNCH(hot_ranks_k, nhot, d_hot, (uint64_t)nhot, rank.p);
    LAUNCH(encode_hot_k, n, d_col, n, rank.p, d_out);
    HIP_OK(hipGetLastError());
    return SPC3D_OK;
}

int localize_device(const DevStream &st, uint64_t n, uint32_t *d_idx, uint32_t *d_ltg,
                    uint32_t *nlocal, std::string &err)
{
    *nlocal = 0;
    if (n == 0)
        return SPC3D_OK;
    if (n >= (1ull << 32)) {
        err = "more than 2^32 - 1 indices are not supported";
        return SPC3D_ERR_TOO_LARGE;
    }
    Arena arena(st);
    HIP_OK(arena.reserve((size_t)n * 44 + ((size_t)8 << 20))); // ten arrays of at most n + 1, scratch
    Temp tmp(arena);
    SBuf<uint32_t> ident, key, pos, head, run_of;
    HIP_OK(ident.alloc(arena, n));
    HIP_OK(key.alloc(arena, n));
    HIP_OK(pos.alloc(arena, n));
    HIP_OK(head.alloc(arena, n + 1));
    HIP_OK(run_of.alloc(arena, n + 1));
    LAUNCH(iota_k, n, ident.p, n);
    TRY(sort_pairs<uint32_t>(tmp, d_idx, key.p, ident.p, pos.p, (uint32_t)n, 32, false, st, err));
    LAUNCH(heads_k, n + 1, key.p, n, head.p);
    TRY(exclusive_sum(tmp, head.p, run_of.p, (size_t)n + 1, st, err));
    uint32_t nruns = 0;
    TRY(fetch(st, &nruns, run_of.p + n, sizeof nruns, err));

    SBuf<uint32_t> first_pos, run_key, first_sorted, run_order, rank_of;
    HIP_OK(first_pos.alloc(arena, nruns));
    HIP_OK(run_key.alloc(arena, nruns));
    HIP_OK(first_sorted.alloc(arena, nruns));
    HIP_OK(run_order.alloc(arena, nruns));
    HIP_OK(rank_of.alloc(arena, nruns));
    // run_of[i] of a head is its run's index; of the other members it is one more
    LAUNCH(run_firsts_k, n, key.p, pos.p, head.p, run_of.p, n, first_pos.p, run_key.p);
    LAUNCH(iota_k, nruns, ident.p, (uint64_t)nruns);
    TRY(sort_pairs<uint32_t>(tmp, first_pos.p, first_sorted.p, ident.p, run_order.p, nruns,
                             bits_for(n - 1), false, st, err));
    LAUNCH(run_ranks_k, nruns, run_order.p, run_key.p, (uint64_t)nruns, rank_of.p, d_ltg);
    LAUNCH(write_local_k, n, pos.p, head.p, run_of.p, rank_of.p, n, d_idx);
    HIP_OK(hipGetLastError());
    HIP_OK(hipStreamSynchronize(st));
    *nlocal = nruns;
    return SPC3D_OK;
}

int remap_device(const DevStream &st, uint64_t n, uint32_t *d_idx, const uint32_t *d_map,
                 uint32_t map_len, std::string &err)
{
    if (n == 0)
        return SPC3D_OK;
    if (n >= (1ull << 32)) {
        err = "more than 2^32 - 1 indices are not supported";
        return SPC3D_ERR_TOO_LARGE;
    }
    DBuf<Counters> dC;
    Counters hC;
    HIP_OK(dC.alloc(st, 1));
    HIP_OK(hipMemsetAsync(dC.p, 0xFF, sizeof(Counters), st));
    // the check and the change queued together: one wait for both
    LAUNCH(remap_check_k, n, d_idx, n, map_len, dC.p);
    LAUNCH(remap_apply_k, n, d_idx, n, d_map, dC.p);
    TRY(fetch(st, &hC, dC.p, sizeof hC, err));
    if (hC.first_bad != 0xFFFFFFFFu) {
        uint32_t v = 0;
        TRY(fetch(st, &v, d_idx + hC.first_bad, sizeof v, err));
        char buf[128];
        std::snprintf(buf, sizeof buf, "index %llu = %u is outside the map of %u entries",
                      (unsigned long long)hC.first_bad, v, map_len);
        err = buf;
        return SPC3D_ERR_BAD_INDEX;
    }
    return SPC3D_OK;
}

} // namespace spc3d

namespace spc3d {

int partition_by_col_block(const DevStream &st, uint64_t nnz, const uint32_t *d_ii, const uint32_t *d_jj,
                           uint32_t ncols, uint32_t nblocks, uint32_t *d_ii_out, uint32_t *d_jj_out,
                           uint32_t *d_order, uint32_t *first, std::string &err)
{
    for (uint32_t b = 0; b <= nblocks; ++b)
        first[b] = 0;
    if (nnz == 0 || nblocks == 0)
        return SPC3D_OK;
    const uint32_t block_cols = (ncols + nblocks - 1) / nblocks;
    Arena arena(st);
    HIP_OK(arena.reserve((size_t)nnz * 12 + (size_t)nblocks * 4 + ((size_t)8 << 20)));
    Temp tmp(arena);
    SBuf<uint32_t> key, key_out, ident, dfirst;
    HIP_OK(key.alloc(arena, nnz));
    HIP_OK(key_out.alloc(arena, nnz));
    HIP_OK(ident.alloc(arena, nnz));
    HIP_OK(dfirst.alloc(arena, (size_t)nblocks + 1));
    LAUNCH(block_keys_k, nnz, d_jj, nnz, block_cols, key.p);
    LAUNCH(iota_k, nnz, ident.p, nnz);
    TRY(sort_pairs<uint32_t>(tmp, key.p, key_out.p, ident.p, d_order, (uint32_t)nnz,
                             bits_for(nblocks), false, st, err));
    LAUNCH(gather_u32_k, nnz, d_ii, d_order, nnz, d_ii_out);
    LAUNCH(gather_u32_k, nnz, d_jj, d_order, nnz, d_jj_out);
    LAUNCH(block_firsts_k, nnz + 1, key_out.p, nnz, nblocks, dfirst.p);
    TRY(fetch(st, first, dfirst.p, ((size_t)nblocks + 1) * sizeof(uint32_t), err));
    return SPC3D_OK;
}

int compose_perm_device(const DevStream &st, const uint32_t *d_order, const uint32_t *d_perm, uint64_t n,
                        uint32_t *d_out, std::string &err)
{
    if (n == 0)
        return SPC3D_OK;
    LAUNCH(compose_perm_k, n, d_order, d_perm, n, d_out);
    HIP_OK(hipGetLastError());
    return SPC3D_OK;
}

int scatter_device(const DevStream &st, const uint32_t *d_perm, const uint32_t *d_vals, uint64_t n,
                   uint32_t *d_out, std::string &err)
{
    if (n == 0)
        return SPC3D_OK;
    LAUNCH(scatter_u32_k, n, d_perm, d_vals, n, d_out);
    HIP_OK(hipGetLastError());
    return SPC3D_OK;
}

int tile_keys_device(const DevStream &st, const uint32_t *d_rows, const uint32_t *d_perm, uint64_t n,
                     uint32_t rows_per_tile, uint32_t *d_key, std::string &err)
{
    if (n == 0)
        return SPC3D_OK;
    LAUNCH(tile_keys_k, n, d_rows, d_perm, n, rows_per_tile, d_key);
    HIP_OK(hipGetLastError());
    return SPC3D_OK;
}

int stable_ranks_device(const DevStream &st, const uint32_t *d_key, uint64_t n, uint32_t max_key,
                        uint32_t *d_rank, std::string &err)
{
    if (n == 0)
        return SPC3D_OK;
    Arena arena(st);
    HIP_OK(arena.reserve((size_t)n * 12 + ((size_t)8 << 20)));
    Temp tmp(arena);
    SBuf<uint32_t> key_out, ident, sorted;
    HIP_OK(key_out.alloc(arena, n));
    HIP_OK(ident.alloc(arena, n));
    HIP_OK(sorted.alloc(arena, n));
    LAUNCH(iota_k, n, ident.p, n);
    TRY(sort_pairs<uint32_t>(tmp, d_key, key_out.p, ident.p, sorted.p, (uint32_t)n,
                             bits_for(max_key), false, st, err));
    LAUNCH(ranks_k, n, sorted.p, n, d_rank);
    HIP_OK(hipGetLastError());
    HIP_OK(hipStreamSynchronize(st)); // the arena goes away with this call
    return SPC3D_OK;
}

// 16 lanes per segment, four entries of a lane in flight: flag[p] = 1 for every entry of a segment
// whose caller's positions are not perm[start], perm[start] + 1, ...
constexpr uint32_t kFlagLanes = 16;
__global__ void staged_flags_k(const Seg *__restrict__ segs, uint32_t nseg,
                               const uint32_t *__restrict__ perm, uint8_t *__restrict__ flag)
{
    const uint32_t sub = threadIdx.x % kFlagLanes;
    GRID_STRIDE(t, (uint64_t)nseg * kFlagLanes) // a group's lanes go round together
    {
        const Seg sg = segs[t / kFlagLanes];
        const uint32_t base = sg.len ? perm[sg.start] : 0;
        bool bad = false;
        for (uint32_t u = sub; u < sg.len; u += 4 * kFlagLanes) {
            uint32_t p[4];
#pragma unroll
            for (uint32_t v = 0; v < 4; ++v)
                p[v] = u + v * kFlagLanes < sg.len ? perm[sg.start + u + v * kFlagLanes]
                                                   : base + u + v * kFlagLanes;
#pragma unroll
            for (uint32_t v = 0; v < 4; ++v)
                bad |= p[v] != base + u + v * kFlagLanes;
        }
        const uint8_t any =
            (__ballot(bad) >> (threadIdx.x & 63u & ~(kFlagLanes - 1))) & ((1ull << kFlagLanes) - 1) ? 1 : 0;
        for (uint32_t u = sub; u < sg.len; u += kFlagLanes)
            flag[sg.start + u] = any;
    }
}

// Numbers for what is marked of n items, in their order: every tile of kMarkTile items counted (count_marks_k),
// a sum over the counts, then a tile's own (mark_ranks).
constexpr int kMarkRounds = 16;
constexpr uint32_t kMarkTile = kTB * kMarkRounds;
constexpr uint32_t kNoHome = 0xFFFFFFFFu;
__device__ __forceinline__ bool marked(uint8_t v) { return v != 0; }
__device__ __forceinline__ bool marked(uint32_t v) { return v != kNoHome; }

template <typename T> __global__ void count_marks_k(const T *__restrict__ v, uint64_t n, uint32_t *cnt)
{
    const uint64_t base = (uint64_t)blockIdx.x * kMarkTile + threadIdx.x;
    uint32_t c = 0;
#pragma unroll
    for (int u = 0; u < kMarkRounds; ++u)
        c += base + u * kTB < n && marked(v[base + u * kTB]);
    c = block_sum(c);
    if (threadIdx.x == 0) {
        cnt[blockIdx.x] = c;
        if (blockIdx.x == 0)
            cnt[gridDim.x] = 0; // the sum's last word is the total
    }
}
// rank[u]: how many are marked before item u * kTB + threadIdx.x of the tile, from `before` on.
__device__ __forceinline__ void mark_ranks(const bool (&on)[kMarkRounds], uint32_t before, uint32_t (&rank)[kMarkRounds])
{
    constexpr int kWaves = kTB / 64;
    static_assert(kMarkRounds * kWaves == 64, "one count for every lane");
    __shared__ uint32_t part[64];
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
#pragma unroll
    for (int u = 0; u < kMarkRounds; ++u) {
        const unsigned long long m = __ballot(on[u]);
        rank[u] = (uint32_t)__popcll(m & ((1ull << lane) - 1));
        if (lane == 0)
            part[u * kWaves + w] = (uint32_t)__popcll(m);
    }
    __syncthreads();
    if (w == 0) {
        const uint32_t mine = part[lane];
        uint32_t upto = mine;
        for (uint32_t d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(upto, d, 64);
            upto += lane >= d ? o : 0u;
        }
        part[lane] = before + upto - mine;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kMarkRounds; ++u)
        rank[u] += part[u * kWaves + w];
}

// A staged entry's slot is its number among them; home: of every caller's position the slot, or kNoHome.
__global__ void staged_fill_k(const uint32_t *__restrict__ perm, const uint8_t *__restrict__ flag,
                              const uint32_t *__restrict__ before, uint64_t nnz, uint32_t *perm2,
                              uint32_t *home)
{
    const uint64_t base = (uint64_t)blockIdx.x * kMarkTile + threadIdx.x;
    bool on[kMarkRounds];
    uint32_t at[kMarkRounds], slot[kMarkRounds];
#pragma unroll
    for (int u = 0; u < kMarkRounds; ++u) {
        const uint64_t p = base + u * kTB < nnz ? base + u * kTB : nnz - 1;
        on[u] = base + u * kTB < nnz && flag[p];
        at[u] = perm[p];
    }
    mark_ranks(on, before[blockIdx.x], slot);
#pragma unroll
    for (int u = 0; u < kMarkRounds; ++u)
        if (base + u * kTB < nnz) {
            perm2[base + u * kTB] = on[u] ? (uint32_t)nnz + slot[u] : at[u];
            home[at[u]] = on[u] ? slot[u] : kNoHome;
        }
}
// The staged results in the caller's order.  This is a sort of (position, slot) pairs whose keys are all
// different: 10.5 M of 16.8 M positions, rows sorted, 310 us by digits and 60 with home written, counted and packed.
__global__ void staged_order_k(const uint32_t *__restrict__ home, const uint32_t *__restrict__ before, uint64_t nnz,
                               uint32_t *dst, uint32_t *src)
{
    const uint64_t base = (uint64_t)blockIdx.x * kMarkTile + threadIdx.x;
    bool on[kMarkRounds];
    uint32_t slot[kMarkRounds], h[kMarkRounds];
#pragma unroll
    for (int u = 0; u < kMarkRounds; ++u) {
        slot[u] = home[base + u * kTB < nnz ? base + u * kTB : nnz - 1];
        on[u] = base + u * kTB < nnz && marked(slot[u]);
    }
    mark_ranks(on, before[blockIdx.x], h);
#pragma unroll
    for (int u = 0; u < kMarkRounds; ++u)
        if (on[u]) {
            dst[h[u]] = (uint32_t)(base + u * kTB);
            src[h[u]] = slot[u];
        }
}

// How many neighbours follow each other.  Four loads in flight per thread: with one this small grid
// waits, 77 us for 15 M entries.
__global__ void adjacent_k(const uint32_t *__restrict__ sorted, uint64_t n, unsigned long long *acc)
{
    unsigned long long c = 0;
    const uint64_t stride = (uint64_t)gridDim.x * kTB;
    for (uint64_t i = (uint64_t)blockIdx.x * kTB + threadIdx.x; i + 1 < n; i += 4 * stride) {
        uint32_t v[4], w[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint64_t j = i + u * stride < n - 1 ? i + u * stride : i;
            v[u] = sorted[j];
            w[u] = sorted[j + 1];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            c += i + u * stride < n - 1 && w[u] == v[u] + 1;
    }
    c = block_sum(c);
    if (threadIdx.x == 0 && c)
        atomicAdd(acc, c);
}

// 64 times the expected number of results that the final pass reads next to another one of their
// wavefront (src_neighbours_k): those d apart in its order share one of its wavefronts for 64 - d of
// 64 starts.  d is what lies between the caller's positions less what is not staged there, a quarter
// at most where this is asked.
__global__ void near_k(const uint32_t *__restrict__ v, uint64_t n, unsigned long long *acc)
{
    unsigned long long c = 0;
    const uint64_t stride = (uint64_t)gridDim.x * kTB;
    for (uint64_t i = (uint64_t)blockIdx.x * kTB + threadIdx.x; i + 1 < n; i += 4 * stride) {
        uint32_t d[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint64_t j = i + u * stride < n - 1 ? i + u * stride : i;
            d[u] = v[j + 1] > v[j] ? v[j + 1] - v[j] : v[j] - v[j + 1];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            c += i + u * stride < n - 1 && d[u] <= 84 ? 64 - d[u] * 3 / 4 : 0;
    }
    c = block_sum(c);
    if (threadIdx.x == 0 && c)
        atomicAdd(acc, c);
}

// How many of the staged results are read next to another one of the same wavefront of
// the final pass (64 consecutive h): src[h] - 1 is the src of another lane.  Of every `every`-th wavefront's
// (a share is asked for, and 10 M results took 135 us; acc[1]: how many were looked at).
__global__ void src_neighbours_k(const uint32_t *__restrict__ src, uint64_t n, uint32_t every,
                                 unsigned long long *acc)
{
    unsigned long long c = 0, looked = 0;
    const uint64_t nround = (n + (uint64_t)64 * every - 1) / ((uint64_t)64 * every) * 64;
    GRID_STRIDE(i, nround)
    {
        const uint64_t h = i / 64 * 64 * every + i % 64;
        const uint32_t mine = h < n ? src[h] : 0xFFFFFFFFu;
        bool near = false;
        for (int j = 0; j < 64; ++j)
            near |= __shfl(mine, j) + 1 == mine;
        looked += h < n;
        if (h < n && near)
            ++c;
    }
    c = block_sum(c);
    looked = block_sum(looked);
    if (threadIdx.x == 0 && looked) {
        atomicAdd(acc, c);
        atomicAdd(acc + 1, looked);
    }
}

int build_store_staging(const DevStream &st, const Seg *d_segs, uint32_t nseg, const uint32_t *d_perm,
                        uint64_t nnz, StoreStaging &out, std::string &err)
{
    out = StoreStaging();
    if (!d_perm || nnz == 0 || nseg == 0 || nnz >= (1ull << 31))
        return SPC3D_OK;
    Arena arena(st);
    HIP_OK(arena.reserve((size_t)nnz * 6 + ((size_t)8 << 20)));
    Temp tmp(arena);
    const uint32_t ntiles = (uint32_t)((nnz + kMarkTile - 1) / kMarkTile);
    SBuf<uint8_t> flag;
    SBuf<uint32_t> cnt, before, home;
    HIP_OK(flag.alloc(arena, nnz));
    HIP_OK(cnt.alloc(arena, (size_t)ntiles + 1));
    HIP_OK(before.alloc(arena, (size_t)ntiles + 1));
    HIP_OK(hipMemsetAsync(flag.p, 0, (size_t)nnz, st));
    LAUNCH(staged_flags_k, (uint64_t)nseg * kFlagLanes, d_segs, nseg, d_perm, flag.p);
    hipLaunchKernelGGL(count_marks_k<uint8_t>, dim3(ntiles), dim3(kTB), 0, st, flag.p, nnz, cnt.p);
    TRY(exclusive_sum(tmp, cnt.p, before.p, (size_t)ntiles + 1, st, err));
    uint32_t n = 0;
    DBuf<unsigned long long> acc;
    HIP_OK(acc.alloc(st, 4));
    HIP_OK(hipMemsetAsync(acc.p, 0, 4 * sizeof(unsigned long long), st));
    LAUNCH_SMALL(near_k, nnz, d_perm, nnz, acc.p + 3);
    unsigned long long near = 0;
    TRY(fetch_all(st, {{&n, before.p + ntiles, sizeof n}, {&near, acc.p + 3, sizeof near}}, err));
    if (n == 0) {
        out.consecutive = true;
        return SPC3D_OK;
    }
    if (nnz + n >= (1ull << 32))
        return SPC3D_OK;
    // What the last check below would turn down, before the work for it (R-MAT 20 with its rows and
    // columns renumbered)
    if ((uint64_t)n * 4 >= nnz * 3 && near / 32 < n)
        return SPC3D_OK;
    DBuf<uint32_t> perm2, dst, src;
    HIP_OK(perm2.alloc(st, nnz));
    HIP_OK(dst.alloc(st, n));
    HIP_OK(src.alloc(st, n));
    HIP_OK(home.alloc(arena, nnz));
    hipLaunchKernelGGL(staged_fill_k, dim3(ntiles), dim3(kTB), 0, st, d_perm, flag.p, before.p, nnz, perm2.p, home.p);
    hipLaunchKernelGGL(count_marks_k<uint32_t>, dim3(ntiles), dim3(kTB), 0, st, home.p, nnz, cnt.p);
    TRY(exclusive_sum(tmp, cnt.p, before.p, (size_t)ntiles + 1, st, err));
    hipLaunchKernelGGL(staged_order_k, dim3(ntiles), dim3(kTB), 0, st, home.p, before.p, nnz, dst.p, src.p);
    // The final pass pays when it writes runs and reads near what its neighbours read; an
    // arbitrary order of the entries gives neither, and keeps its scattered stores.
    LAUNCH_SMALL(adjacent_k, n, dst.p, (uint64_t)n, acc.p);
    const uint32_t every = n >= (1u << 20) ? 16 : 1;
    LAUNCH_SMALL(src_neighbours_k, n / every + 1, src.p, (uint64_t)n, every, acc.p + 1);
    unsigned long long seen[3] = {0, 0, 0};
    TRY(fetch(st, seen, acc.p, sizeof seen, err));
    if (seen[0] * 2 < n || seen[1] * 2 < seen[2])
        return SPC3D_OK; // (the DBufs free themselves)
    out.perm2 = perm2.release();
    out.dst = dst.release();
    out.src = src.release();
    out.n = n;
    out.consecutive = true;
    return SPC3D_OK;
}

__global__ void quotients_k(const uint32_t *__restrict__ v, uint64_t n, uint32_t T, uint32_t *out)
{
    GRID_STRIDE(p, n) out[p] = v[p] / T;
}

__global__ void two_pass_mid_k(const uint32_t *__restrict__ sp2, const uint32_t *__restrict__ perm,
                               uint64_t n, uint32_t T, uint32_t *mid_of, uint16_t *l2)
{
    GRID_STRIDE(m, n)
    {
        const uint32_t p = sp2[m];
        mid_of[p] = (uint32_t)m;
        l2[perm[p]] = (uint16_t)(m % T);
    }
}

__global__ void two_pass_slots_k(const uint32_t *__restrict__ sp1,
                                 const uint32_t *__restrict__ mid_of, uint64_t n, uint32_t T,
                                 uint16_t *l1, uint32_t *dst1)
{
    GRID_STRIDE(s, n)
    {
        const uint32_t p = sp1[s];
        l1[s] = (uint16_t)(p - (uint32_t)(s / T) * T); // the sort kept every tile in its place
        dst1[s] = mid_of[p];
    }
}

// The same tables without sorts, for up to kCountedTiles tiles: how many elements every tile has for
// every bucket (count), where each such run starts in the intermediate vector (a scan in bucket order),
// then one more pass that draws an element's place in its run from LDS counters.  Inside a run the
// elements come as they are drawn: any order serves, the three tables agree on it.  16 M entries in
// arbitrary order, fp64: two sorts and their passes 850 us, this 165.  The line: two counters per bucket
// and the partial sums within 64 KiB of LDS (157 M fp64 results); the two tables of counts, 8 bytes per
// pair of tiles, are then under a fifth of what the sorts need.
constexpr uint32_t kCountedTiles = 7680;
constexpr int kTwoPassTB = 1024;

__global__ void __launch_bounds__(kTwoPassTB)
two_pass_count_k(const uint32_t *__restrict__ perm, uint64_t n, uint32_t T, uint32_t nt,
                 uint32_t *__restrict__ count)
{
    extern __shared__ uint32_t words[];
    for (uint32_t b = threadIdx.x; b < nt; b += kTwoPassTB)
        words[b] = 0;
    __syncthreads();
    const uint64_t lo = (uint64_t)blockIdx.x * T, hi = lo + T < n ? lo + T : n;
    for (uint64_t p = lo + threadIdx.x; p < hi; p += kTwoPassTB)
        atomicAdd(&words[perm[p] / T], 1u);
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < nt; b += kTwoPassTB)
        count[(uint64_t)b * nt + blockIdx.x] = words[b];
}

// start: the exclusive sums of count, bucket by bucket, inside a bucket tile by tile.
__global__ void __launch_bounds__(kTwoPassTB)
two_pass_place_k(const uint32_t *__restrict__ perm, uint64_t n, uint32_t T, uint32_t nt,
                 const uint32_t *__restrict__ count, const uint32_t *__restrict__ start,
                 uint16_t *__restrict__ l1, uint32_t *__restrict__ dst1, uint16_t *__restrict__ l2)
{
    extern __shared__ uint32_t words[];
    __shared__ uint32_t part[kTwoPassTB];
    uint32_t *next = words, *shift = words + nt; // the run's next slot in the tile; its place - its slot
    // slots of the tile's runs: exclusive sums over the buckets, a stretch of them per thread
    const uint32_t per = (nt + kTwoPassTB - 1) / kTwoPassTB;
    const uint32_t b0 = threadIdx.x * per < nt ? threadIdx.x * per : nt, b1 = b0 + per < nt ? b0 + per : nt;
    uint32_t sum = 0;
    for (uint32_t b = b0; b < b1; ++b)
        sum += count[(uint64_t)b * nt + blockIdx.x];
    part[threadIdx.x] = sum;
    __syncthreads();
    for (uint32_t step = 1; step < kTwoPassTB; step *= 2) {
        const uint32_t add = threadIdx.x >= step ? part[threadIdx.x - step] : 0;
        __syncthreads();
        part[threadIdx.x] += add;
        __syncthreads();
    }
    uint32_t slot = part[threadIdx.x] - sum;
    for (uint32_t b = b0; b < b1; ++b) {
        next[b] = slot;
        shift[b] = start[(uint64_t)b * nt + blockIdx.x] - slot;
        slot += count[(uint64_t)b * nt + blockIdx.x];
    }
    __syncthreads();
    const uint64_t lo = (uint64_t)blockIdx.x * T, hi = lo + T < n ? lo + T : n;
    for (uint64_t p = lo + threadIdx.x; p < hi; p += kTwoPassTB) {
        const uint32_t e = perm[p], b = e / T;
        const uint32_t s = atomicAdd(&next[b], 1u), m = s + shift[b];
        l1[lo + s] = (uint16_t)(p - lo);
        dst1[lo + s] = m;
        l2[e] = (uint16_t)(m - b * T);
    }
}

int build_two_pass(const DevStream &st, const uint32_t *d_perm, uint64_t nnz, uint32_t T, TwoPass &out,
                   std::string &err)
{
    out = TwoPass();
    if (!d_perm || T == 0 || T > 65536 || nnz >= (1ull << 32) || nnz < 2ull * T)
        return SPC3D_OK;
    const uint64_t ntiles64 = (nnz + T - 1) / T;
    if (ntiles64 * ntiles64 >= (1ull << 32))
        return SPC3D_OK;
    Arena arena(st);
    DBuf<uint16_t> l1, l2;
    DBuf<uint32_t> dst1;
    HIP_OK(l1.alloc(st, nnz));
    HIP_OK(l2.alloc(st, nnz));
    HIP_OK(dst1.alloc(st, nnz));
    if (ntiles64 <= kCountedTiles) {
        const uint32_t nt = (uint32_t)ntiles64;
        const size_t runs = (size_t)nt * nt;
        HIP_OK(arena.reserve(runs * 8 + ((size_t)8 << 20)));
        Temp tmp(arena);
        SBuf<uint32_t> count, start;
        HIP_OK(count.alloc(arena, runs));
        HIP_OK(start.alloc(arena, runs));
        hipLaunchKernelGGL(two_pass_count_k, dim3(nt), dim3(kTwoPassTB), nt * sizeof(uint32_t), st, d_perm,
                           nnz, T, nt, count.p);
        TRY(exclusive_sum(tmp, count.p, start.p, runs, st, err));
        hipLaunchKernelGGL(two_pass_place_k, dim3(nt), dim3(kTwoPassTB), 2 * nt * sizeof(uint32_t), st,
                           d_perm, nnz, T, nt, count.p, start.p, l1.p, dst1.p, l2.p);
        HIP_OK(hipGetLastError());
        HIP_OK(hipStreamSynchronize(st));
        out.l1 = l1.release();
        out.l2 = l2.release();
        out.dst1 = dst1.release();
        out.tile = T;
        out.n = nnz;
        return SPC3D_OK;
    }
    HIP_OK(arena.reserve((size_t)nnz * 20 + ((size_t)8 << 20)));
    Temp tmp(arena);
    SBuf<uint32_t> key, idx, key_out, sp1, sp2, mid_of;
    HIP_OK(key.alloc(arena, nnz));
    HIP_OK(idx.alloc(arena, nnz));
    HIP_OK(key_out.alloc(arena, nnz));
    HIP_OK(sp1.alloc(arena, nnz));
    HIP_OK(sp2.alloc(arena, nnz));
    // Kernel positions by bucket of the caller's position, inside a bucket by tile (their own order,
    // the sorts being stable); then those by tile, inside a tile by bucket.  Keys of one number each:
    // of (tile, bucket) pairs both sorts took half as many passes again.
    const int bits = bits_for(ntiles64 - 1);
    LAUNCH(quotients_k, nnz, d_perm, nnz, T, key.p);
    LAUNCH(iota_k, nnz, idx.p, nnz);
    TRY(sort_pairs<uint32_t>(tmp, key.p, key_out.p, idx.p, sp2.p, (uint32_t)nnz, bits, false, st, err));
    LAUNCH(quotients_k, nnz, sp2.p, nnz, T, key.p);
    TRY(sort_pairs<uint32_t>(tmp, key.p, key_out.p, sp2.p, sp1.p, (uint32_t)nnz, bits, false, st, err));
    mid_of.p = key.p; // the keys are no longer needed
    LAUNCH(two_pass_mid_k, nnz, sp2.p, d_perm, nnz, T, mid_of.p, l2.p);
    LAUNCH(two_pass_slots_k, nnz, sp1.p, mid_of.p, nnz, T, l1.p, dst1.p);
    HIP_OK(hipGetLastError());
    HIP_OK(hipStreamSynchronize(st));
    out.l1 = l1.release();
    out.l2 = l2.release();
    out.dst1 = dst1.release();
    out.tile = T;
    out.n = nnz;
    return SPC3D_OK;
}

// ---- row tiles x column blocks ("sweep") ---------------------------------------------
// out[perm[q]] = base + q
__global__ void inverse_offsets_k(const uint32_t *__restrict__ perm, uint64_t n, uint32_t base,
                                  uint32_t *out)
{
    GRID_STRIDE(q, n) out[perm[q]] = base + (uint32_t)q;
}

// Rows of at least `least` entries.
__global__ void count_min_k(const uint32_t *__restrict__ cnt, uint64_t nrows, uint32_t least,
                            unsigned long long *out)
{
    unsigned long long c = 0;
    GRID_STRIDE(r, nrows) c += cnt[r] >= least;
    c = block_sum(c);
    if (threadIdx.x == 0 && c)
        atomicAdd(out, c);
}

// key[j] = (generation of rank j) << 32 | row of rank j
__global__ void sweep_gen_keys_k(const uint32_t *__restrict__ order, uint32_t nin, uint64_t per_gen,
                                 unsigned long long *key)
{
    GRID_STRIDE(j, nin) key[j] = ((unsigned long long)(j / per_gen) << 32) | order[j];
}

// Tile and local row of the j-th row of the sweep (by generation, inside a generation by row
// number): rpt consecutive rows make a tile (rpt_last in the last generation).
__global__ void sweep_rows_k(const unsigned long long *__restrict__ gen_row, uint32_t nin,
                             uint32_t P, uint32_t R, uint32_t last_gen, uint32_t rpt_last,
                             uint32_t *row_tile, uint32_t *row_local, uint32_t *tile_rows)
{
    GRID_STRIDE(j, nin)
    {
        const uint32_t row = (uint32_t)gen_row[j];
        const uint64_t per_gen = (uint64_t)P * R;
        const uint32_t gen = (uint32_t)(j / per_gen), jl = (uint32_t)(j % per_gen);
        const uint32_t rpt = gen == last_gen ? rpt_last : R;
        const uint32_t t = gen * P + jl / rpt, l = jl % rpt;
        row_tile[row] = t;
        row_local[row] = l;
        tile_rows[(uint64_t)t * R + l] = row;
    }
}

// Sort key of entry e: (tile, block, local row); one past the largest such key for an entry
// of a row outside the sweep (they sort last, in the caller's order).
template <typename KeyT>
__global__ void sweep_keys_k(const uint32_t *__restrict__ ii, const uint32_t *__restrict__ jj,
                             uint64_t nnz, const uint32_t *__restrict__ row_tile,
                             const uint32_t *__restrict__ row_local, uint32_t block_cols,
                             uint32_t nb, uint32_t R, KeyT rest_key, KeyT *key,
                             unsigned long long *nin)
{
    unsigned long long mine = 0;
    GRID_STRIDE(e, nnz)
    {
        const uint32_t r = ii[e], t = row_tile[r];
        if (t == 0xFFFFFFFFu) {
            key[e] = rest_key;
            continue;
        }
        key[e] = ((KeyT)t * nb + jj[e] / block_cols) * R + row_local[r];
        ++mine;
    }
    mine = block_sum(mine);
    if (threadIdx.x == 0 && mine)
        atomicAdd(nin, mine);
}

// Of the sorted sweep entries: column, local row, and the (tile, block) bin.
template <typename KeyT>
__global__ void sweep_entries_k(const KeyT *__restrict__ skey,
                                const uint32_t *__restrict__ perm,
                                const uint32_t *__restrict__ jj, uint64_t n, uint32_t R,
                                uint32_t *col, uint16_t *lrow, uint32_t *bin)
{
    GRID_STRIDE(k, n)
    {
        const KeyT key = skey[k];
        bin[k] = (uint32_t)(key / R);
        lrow[k] = (uint16_t)(key % R);
        col[k] = jj[perm[k]];
    }
}

// The entries in sweep order: perm (all nnz, those outside the sweep last), and column, local row
// and bin of the n inside.
template <typename KeyT>
int sweep_entries(Arena &arena, Temp &tmp, const DevStream &st, uint64_t nnz, const uint32_t *d_ii,
                  const uint32_t *d_jj, const uint32_t *row_tile, const uint32_t *row_local,
                  uint32_t block_cols, uint32_t nb, uint32_t R, KeyT rest_key, unsigned long long *d_n,
                  DBuf<uint32_t> &perm, DBuf<uint32_t> &col, DBuf<uint16_t> &lrow, SBuf<uint32_t> &bin,
                  uint64_t &n, std::string &err)
{
    SBuf<KeyT> key, skey;
    SBuf<uint32_t> ident;
    HIP_OK(key.alloc(arena, nnz));
    HIP_OK(skey.alloc(arena, nnz));
    HIP_OK(ident.alloc(arena, nnz));
    HIP_OK(perm.alloc(st, nnz));
    LAUNCH_SMALL((sweep_keys_k<KeyT>), nnz, d_ii, d_jj, nnz, row_tile, row_local, block_cols, nb, R,
                 rest_key, key.p, d_n);
    LAUNCH(iota_k, nnz, ident.p, nnz);
    TRY(sort_pairs<KeyT>(tmp, key.p, skey.p, ident.p, perm.p, (uint32_t)nnz, bits_for(rest_key), false,
                         st, err));
    unsigned long long seen = 0;
    TRY(fetch(st, &seen, d_n, sizeof seen, err));
    n = seen;
    if (n == 0)
        return SPC3D_OK;
    HIP_OK(col.alloc(st, n));
    HIP_OK(lrow.alloc(st, n));
    HIP_OK(bin.alloc(arena, n));
    LAUNCH((sweep_entries_k<KeyT>), n, skey.p, perm.p, d_jj, n, R, col.p, lrow.p, bin.p);
    HIP_OK(hipGetLastError());
    return SPC3D_OK;
}

int build_sweep(const DevStream &st, uint32_t nrows, uint32_t ncols, uint64_t nnz, const uint32_t *d_ii,
                const uint32_t *d_jj, uint32_t lanes, uint32_t R, uint32_t nb, uint32_t min_row,
                uint32_t P, SweepPlan &out, std::string &err)
{
    out = SweepPlan();
    if (nnz == 0 || nnz >= (1ull << 32) || lanes == 0 || R == 0 || R > 65536 || nb == 0 || P == 0)
        return SPC3D_OK;
    const uint32_t G = 1024 / lanes;
    if (G == 0)
        return SPC3D_OK;
    const uint32_t block_cols = (ncols + nb - 1) / nb;
    Arena arena(st);
    HIP_OK(arena.reserve(((size_t)nrows + 1) * 40 + (size_t)nnz * 36 + ((size_t)8 << 20)));
    Temp tmp(arena);
    // ---- rows by length ----
    SBuf<uint32_t> rowcnt, rowid, order, cnt_sorted, row_tile, row_local;
    SBuf<unsigned long long> total, gkey, gkey_sorted;
    HIP_OK(rowcnt.alloc(arena, (size_t)nrows + 1));
    HIP_OK(rowid.alloc(arena, nrows));
    HIP_OK(order.alloc(arena, nrows));
    HIP_OK(cnt_sorted.alloc(arena, nrows));
    HIP_OK(row_tile.alloc(arena, nrows));
    HIP_OK(row_local.alloc(arena, nrows));
    HIP_OK(total.alloc(arena, 1));
    HIP_OK(hipMemsetAsync(rowcnt.p, 0, ((size_t)nrows + 1) * sizeof(uint32_t), st));
    HIP_OK(hipMemsetAsync(total.p, 0, sizeof(unsigned long long), st));
    // one addition per run of equal row numbers inside a wavefront: few for rows that arrive
    // together, one per entry at worst
    LAUNCH(hist_sorted_k, nnz, d_ii, nnz, rowcnt.p);
    // rows by length, longest first, equal lengths in row order; those of at least min_row
    // entries come first and are the sweep's
    LAUNCH(iota_k, nrows, rowid.p, (uint64_t)nrows);
    TRY(sort_pairs<uint32_t>(tmp, rowcnt.p, cnt_sorted.p, rowid.p, order.p, nrows, 32, true, st, err));
    LAUNCH_SMALL(count_min_k, nrows, rowcnt.p, nrows, std::max(1u, min_row), total.p);
    unsigned long long seen = 0;
    TRY(fetch(st, &seen, total.p, sizeof seen, err));
    HIP_OK(hipMemsetAsync(total.p, 0, sizeof(unsigned long long), st));
    const uint32_t nin = (uint32_t)seen;
    if (nin == 0)
        return SPC3D_OK;
    // A generation: the next P * R rows by length, which one launch of P tiles takes.  Inside
    // a generation the rows are of similar length, and a tile takes R of them that are
    // consecutive by row number: the tiles of a launch stay level to about a percent, and
    // what a tile reads and writes (its rows of A or Y, its SDDMM results on their way to
    // the caller's order) lies together.  The last generation spreads its rows over the P
    // tiles.
    const uint64_t per_gen = (uint64_t)P * R;
    const uint64_t gens = (nin + per_gen - 1) / per_gen;
    const uint64_t last = nin - (gens - 1) * per_gen; // rows of the last generation
    const uint32_t rpt_last = (uint32_t)((last + P - 1) / P);
    const uint64_t ntiles64 = (gens - 1) * P + (last + rpt_last - 1) / rpt_last;
    if (ntiles64 * nb + 1 >= (1ull << 32))
        return SPC3D_OK;
    const uint32_t ntiles = (uint32_t)ntiles64;
    HIP_OK(gkey.alloc(arena, nin));
    HIP_OK(gkey_sorted.alloc(arena, nin));
    LAUNCH(sweep_gen_keys_k, nin, order.p, nin, per_gen, gkey.p);
    // (values unused: cnt_sorted and rowid are free by now)
    TRY(sort_pairs<unsigned long long>(tmp, gkey.p, gkey_sorted.p, rowid.p, cnt_sorted.p, nin,
                                       32 + bits_for(gens), false, st, err));
    DBuf<uint32_t> tile_rows, perm, col, ptr;
    DBuf<uint16_t> lrow;
    HIP_OK(tile_rows.alloc(st, (size_t)ntiles * R));
    HIP_OK(hipMemsetAsync(tile_rows.p, 0xFF, (size_t)ntiles * R * sizeof(uint32_t), st));
    HIP_OK(hipMemsetAsync(row_tile.p, 0xFF, (size_t)nrows * sizeof(uint32_t), st));
    LAUNCH(sweep_rows_k, nin, gkey_sorted.p, nin, P, R, (uint32_t)(gens - 1), rpt_last, row_tile.p,
           row_local.p, tile_rows.p);
    // ---- entries ----
    SBuf<uint32_t> bin;
    const uint64_t nbins = (uint64_t)ntiles * nb;
    const unsigned long long rest_key = (unsigned long long)nbins * R;
    uint64_t n = 0;
    if (rest_key >> 32)
        TRY(sweep_entries<unsigned long long>(arena, tmp, st, nnz, d_ii, d_jj, row_tile.p, row_local.p,
                                              block_cols, nb, R, rest_key, total.p, perm, col, lrow, bin, n, err));
    else // half the keys' traffic in the sort
        TRY(sweep_entries<uint32_t>(arena, tmp, st, nnz, d_ii, d_jj, row_tile.p, row_local.p, block_cols,
                                    nb, R, (uint32_t)rest_key, total.p, perm, col, lrow, bin, n, err));
    if (n == 0)
        return SPC3D_OK;
    HIP_OK(ptr.alloc(st, nbins + 1));
    SBuf<uint32_t> bstart, bcnt;
    HIP_OK(bstart.alloc(arena, nbins));
    HIP_OK(bcnt.alloc(arena, nbins + 1));
    HIP_OK(hipMemsetAsync(bcnt.p, 0, (nbins + 1) * sizeof(uint32_t), st));
    LAUNCH(run_bounds_k, n, bin.p, n, (uint32_t)nbins, bstart.p, bcnt.p);
    LAUNCH(run_lengths_k, nbins, bstart.p, nbins, bcnt.p);
    TRY(exclusive_sum(tmp, bcnt.p, ptr.p, (size_t)nbins + 1, st, err));
    HIP_OK(hipGetLastError());
    HIP_OK(hipStreamSynchronize(st));
    out.perm = perm.release();
    out.col = col.release();
    out.lrow = lrow.release();
    out.ptr = ptr.release();
    out.tile_rows = tile_rows.release();
    out.n = n;
    out.ntiles = ntiles;
    out.nblocks = nb;
    out.rows_per_tile = R;
    out.groups = G;
    out.lanes = lanes;
    out.per_launch = P;
    out.nrows_in = nin;
    return SPC3D_OK;
}

// ---- row tiles over skewed columns ----------------------------------------------------
struct HubCounters {
    uint32_t nsplit, nslots; // cut rows; partial-sum rows, gaps included
    uint32_t left_out;       // segments of rows without a place that need one
    uint32_t rest[kSlices];  // segments of other rows per queue
    uint32_t adjacent;       // entries of a tile that follow their predecessor in the caller's order too (at least)
};

// What the scan adds up: [0, ncols] how much of an L2 a column takes on average, in 1/1024 of its dense row (the
// tiles of an XCD are an eighth of all, and meet a column of d entries with probability 1 - (7/8)^d); and from
// ncols + 1 on, per row of at least min_row entries, its pieces.  And what starts as nothing.
__global__ void hub_start_k(const uint32_t *__restrict__ deg, uint64_t ncols, const uint32_t *__restrict__ rowptr,
                            uint64_t nrows, uint32_t min_row, uint32_t cut, uint64_t nplaces, uint32_t *sums,
                            uint8_t *row_in, uint32_t *tile_rows, TilePlace *place, HubCounters *C)
{
    const uint64_t n = ncols + nrows + 2 > nplaces ? ncols + nrows + 2 : nplaces;
    GRID_STRIDE(i, n)
    {
        if (i <= ncols) {
            uint32_t miss = 1024; // of 1024, rounded down at every step
            const uint32_t d = i < ncols ? (deg[i] < 52 ? deg[i] : 52u) : 0u;
            for (uint32_t k = 0; k < d; ++k)
                miss = miss * 7 / 8;
            sums[i] = 1024 - miss;
        } else if (i < ncols + nrows + 2) {
            const uint64_t r = i - ncols - 1;
            const uint32_t len = r < nrows ? rowptr[r + 1] - rowptr[r] : 0u;
            sums[i] = len >= min_row ? (len + cut - 1) / cut : 0u;
            if (r < nrows)
                row_in[r] = 0;
        }
        if (i < nplaces) {
            tile_rows[i] = 0xFFFFFFFFu;
            place[i] = TilePlace{0, 0, 0};
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0)
        *C = HubCounters{};
}
// Of every column its block, and no rank.
__global__ void hub_blocks_k(const uint32_t *__restrict__ before, uint64_t ncols, uint32_t per_block, uint32_t nb,
                             uint16_t *block, uint16_t *rank)
{
    GRID_STRIDE(c, ncols)
    {
        const uint32_t b = before[c] / per_block;
        block[c] = (uint16_t)(b < nb ? b : nb - 1);
        if (rank)
            rank[c] = 0xFFFFu;
    }
}
// The pieces, a row's together, under a sort key that is the length to an eighth of an octave.
__global__ void hub_pieces_k(const uint32_t *__restrict__ rowptr, uint64_t nrows, const uint32_t *__restrict__ first,
                             uint32_t base, uint32_t *key, uint32_t *id, uint32_t *row)
{
    GRID_STRIDE(r, nrows)
    {
        const uint32_t at = first[r] - base, np = first[r + 1] - first[r];
        if (!np)
            continue;
        const uint32_t len = (rowptr[r + 1] - rowptr[r]) / np, e = 31 - __clz((int)len);
        const uint32_t k = e * 8 + (uint32_t)(((unsigned long long)len << 3 >> e) & 7);
        for (uint32_t i = 0; i < np; ++i) {
            key[at + i] = k;
            id[at + i] = at + i;
            row[at + i] = (uint32_t)r;
        }
    }
}

// The piece of rank j (longest first) goes to tile j mod P, there and back.  A cut row's
// pieces have neighbouring ranks; its partial sums are the slots of those numbers.  A row has places for
// all its pieces or for none.
__global__ void hub_places_k(const uint32_t *__restrict__ order, const uint32_t *__restrict__ row_of,
                             uint64_t npc, const uint32_t *__restrict__ rowptr,
                             const uint32_t *__restrict__ first, uint32_t base, uint32_t P,
                             uint32_t R, TilePlace *place, uint32_t *tile_rows, uint32_t *slot,
                             uint8_t *row_in, SplitRow *splits, HubCounters *C)
{
    GRID_STRIDE(j, npc)
    {
        const uint32_t pc = order[j], row = row_of[pc], np = first[row + 1] - first[row], i = pc - (first[row] - base);
        if (j - i + np > (uint64_t)P * R)
            continue;
        const uint32_t l = (uint32_t)j / P, x = (uint32_t)j % P;
        const uint64_t at = (uint64_t)(l & 1 ? P - 1 - x : x) * R + l;
        const uint32_t start = rowptr[row], len = rowptr[row + 1] - start;
        const uint32_t groups = (len + kTileGroup - 1) / kTileGroup, mine = (groups - i + np - 1) / np * kTileGroup;
        place[at] = TilePlace{start + i * kTileGroup, np * kTileGroup,
                              mine - ((groups - 1) % np == i ? groups * kTileGroup - len : 0)};
        tile_rows[at] = row;
        slot[at] = np > 1 ? (uint32_t)j : kWholeRow;
        row_in[row] = 1;
        if (np > 1 && i == 0) {
            splits[atomicAdd(&C->nsplit, 1u)] = SplitRow{row, (uint32_t)j, np, 0};
            atomicMax(&C->nslots, (uint32_t)j + np);
        }
    }
}

// One workgroup per tile: entries before each of its places, and in all.
__global__ void __launch_bounds__(kTileMaxRows)
hub_offsets_k(const TilePlace *__restrict__ place, uint32_t R, uint32_t *off, uint32_t *tile_n)
{
    __shared__ uint32_t sum[kTileMaxRows / 64];
    const uint32_t l = threadIdx.x, lane = l & 63u, wave = l >> 6;
    const uint64_t at = (uint64_t)blockIdx.x * R + l;
    const uint32_t len = l < R ? place[at].len : 0u;
    uint32_t upto = len;
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t v = __shfl_up(upto, d, 64);
        upto += lane >= d ? v : 0u;
    }
    if (lane == 63)
        sum[wave] = upto;
    __syncthreads();
    uint32_t total = 0, before = 0;
    for (uint32_t w = 0; w < kTileMaxRows / 64; ++w) {
        before += w < wave ? sum[w] : 0u;
        total += sum[w];
    }
    if (l < R)
        off[at] = before + upto - len;
    if (l == 0)
        tile_n[blockIdx.x] = total;
}

// One workgroup per tile: its entries by block, in a block by place, in a place in the order of the source.
// They are counted by block first, then taken in the order of the places, kFillRound at a time: every wavefront
// counts its own by block, a thread per block adds those up, and the wavefronts lay theirs out from there.  All
// wavefronts write near the same few places of every block, so that lines are full when they leave the L2:
// R-MAT 20, 13 M entries, 241 us (266 without a round's loads under way during the one before); 277 with a sixteenth
// of the tile to every wavefront, and 500 for a device-wide radix sort on (tile, block, place) and the gathers after it.
constexpr int kFillTB = 1024;
constexpr uint32_t kFillBlocks = 1027; // at most
struct HubFill {
    const uint32_t *col, *pos; // the source; pos (may be null): caller's position of entry p
    const uint16_t *block, *hot; // of a column: its block, and its rank where it is hot (null: none is)
    const TilePlace *place;
    const uint32_t *off, *tptr;
    uint32_t R, nb;
    bool by_pos; // results go to the caller's position, else to the entry's in the source
    uint32_t *where; // scratch: place << 16 | block of every entry
    uint32_t *ptr, *out_col, *out_perm, *src, *dst;
    uint16_t *lrow;
    HubCounters *C;
};
__device__ __forceinline__ uint32_t place_at(uint32_t start, uint32_t step, uint32_t y)
{
    return start + y / kTileGroup * step + y % kTileGroup;
}
__global__ void __launch_bounds__(kFillTB) hub_fill_k(HubFill F)
{
    constexpr uint32_t kWaves = kFillTB / 64;
    __shared__ uint32_t first[kTileMaxRows + 1], start[kTileMaxRows], step[kTileMaxRows];
    __shared__ uint32_t counts[kWaves * kFillBlocks], next[kFillBlocks];
    const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    volatile uint32_t *count = counts + w * kFillBlocks;
    const uint32_t t = blockIdx.x, lo = F.tptr[t], n = F.tptr[t + 1] - lo;
    for (uint32_t l = threadIdx.x; l <= F.R; l += kFillTB) {
        const uint64_t at = (uint64_t)t * F.R + l;
        first[l] = l < F.R ? F.off[at] : n;
        if (l < F.R) {
            start[l] = F.place[at].start;
            step[l] = F.place[at].step;
        }
    }
    for (uint32_t k = lane; k < F.nb; k += 64)
        count[k] = 0;
    __syncthreads();
    constexpr int V = 8; // entries of a lane at a time, here
    for (uint32_t y0 = w * V * 64; y0 < n; y0 += kWaves * V * 64) {
        // the place of the first, and from there of the others: few places end among 512 entries
        uint32_t at = 0, up = F.R;
        while (up - at > 1) {
            const uint32_t mid = (at + up) / 2;
            if (first[mid] <= y0)
                at = mid;
            else
                up = mid;
        }
        uint32_t l[V], c[V];
#pragma unroll
        for (int u = 0; u < V; ++u) {
            const uint32_t y = y0 + u * 64 + lane < n ? y0 + u * 64 + lane : n - 1;
            l[u] = u ? l[u ? u - 1 : 0] : at;
            while (__any(first[l[u] + 1] <= y)) // (first[R] == n: no lane goes past the last place)
                l[u] += first[l[u] + 1] <= y;
            c[u] = F.col[place_at(start[l[u]], step[l[u]], y - first[l[u]])];
        }
#pragma unroll
        for (int u = 0; u < V; ++u)
            c[u] = F.block[c[u]];
#pragma unroll
        for (int u = 0; u < V; ++u)
            if (y0 + u * 64 + lane < n) {
                atomicAdd(const_cast<uint32_t *>(&count[c[u]]), 1u);
                F.where[lo + y0 + u * 64 + lane] = l[u] << 16 | c[u];
            }
    }
    __syncthreads();
    if (w == 0) { // where the blocks begin
        uint32_t run = 0;
        for (uint32_t k0 = 0; k0 < F.nb; k0 += 64) {
            const uint32_t k = k0 + lane;
            uint32_t sum = 0;
            if (k < F.nb)
                for (uint32_t v = 0; v < kWaves; ++v)
                    sum += counts[v * kFillBlocks + k];
            uint32_t upto = sum;
            for (uint32_t d = 1; d < 64; d <<= 1) {
                const uint32_t o = __shfl_up(upto, d, 64);
                upto += lane >= d ? o : 0u;
            }
            if (k < F.nb) {
                next[k] = run + upto - sum;
                F.ptr[(uint64_t)t * F.nb + k] = lo + run + upto - sum;
            }
            run += __shfl(upto, 63, 64);
        }
        if (lane == 0 && t + 1 == gridDim.x)
            F.ptr[(uint64_t)(t + 1) * F.nb] = lo + n;
    }
    int bits = 1;
    while ((F.nb - 1) >> bits)
        ++bits;
    uint32_t adjacent = 0;
    constexpr int U = 4; // and here
    constexpr uint32_t kFillRound = kWaves * U * 64;
    // The loads of a round are under way while the one before is laid out.
    uint32_t next_at[U], next_col[U], next_pos[U];
    auto where_of = [&](uint32_t r0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t y = r0 + w * U * 64 + u * 64 + lane;
            next_at[u] = F.where[lo + (y < n ? y : n - 1)];
        }
    };
    auto source_of = [&](uint32_t r0, int u) {
        const uint32_t y = r0 + w * U * 64 + u * 64 + lane, l = next_at[u] >> 16;
        return place_at(start[l], step[l], (y < n ? y : n - 1) - first[l]);
    };
    if (n) {
        where_of(0);
#pragma unroll
        for (int u = 0; u < U; ++u)
            next_col[u] = F.col[source_of(0, u)];
        if (F.pos)
#pragma unroll
            for (int u = 0; u < U; ++u)
                next_pos[u] = F.pos[source_of(0, u)];
    }
    for (uint32_t r0 = 0; r0 < n; r0 += kFillRound) {
        const uint32_t y0 = r0 + w * U * 64;
        uint32_t l[U], p[U], c[U], h[U], blk[U], e[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            p[u] = source_of(r0, u);
            l[u] = next_at[u] >> 16;
            blk[u] = next_at[u] & 0xFFFFu;
            c[u] = next_col[u];
            e[u] = F.pos ? next_pos[u] : p[u];
            h[u] = F.hot ? F.hot[c[u]] : 0xFFFFu;
        }
        const bool more = r0 + kFillRound < n;
        if (more)
            where_of(r0 + kFillRound);
        __syncthreads(); // the round before has laid its entries out (the first: the blocks' beginnings are there)
        for (uint32_t k = lane; k < F.nb; k += 64)
            count[k] = 0;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (y0 + u * 64 + lane < n)
                atomicAdd(const_cast<uint32_t *>(&count[blk[u]]), 1u);
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < F.nb; k += kFillTB) {
            uint32_t m[kWaves], at = next[k];
#pragma unroll
            for (uint32_t v = 0; v < kWaves; ++v)
                m[v] = counts[v * kFillBlocks + k];
#pragma unroll
            for (uint32_t v = 0; v < kWaves; ++v) {
                counts[v * kFillBlocks + k] = at;
                at += m[v];
            }
            next[k] = at;
        }
        if (more) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                next_col[u] = F.col[source_of(r0 + kFillRound, u)];
            if (F.pos)
#pragma unroll
                for (int u = 0; u < U; ++u)
                    next_pos[u] = F.pos[source_of(r0 + kFillRound, u)];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool on = y0 + u * 64 + lane < n;
            const uint32_t e0 = __shfl_up(e[u], 1, 64), blk0 = __shfl_up(blk[u], 1, 64);
            adjacent += (uint32_t)__popcll(__ballot(on && lane && e0 + 1 == e[u] && blk0 == blk[u]));
            unsigned long long same = __ballot(on); // lanes with an entry of this block
            for (int k = 0; k < bits; ++k) {
                const unsigned long long m = __ballot((blk[u] >> k & 1) != 0);
                same &= (blk[u] >> k & 1) ? m : ~m;
            }
            if (on) {
                const uint32_t rank = (uint32_t)__popcll(same & ((1ull << lane) - 1));
                const uint32_t base = count[blk[u]];
                if (rank == 0)
                    count[blk[u]] = base + (uint32_t)__popcll(same);
                const uint32_t at = lo + base + rank;
                F.out_col[at] = h[u] == 0xFFFFu ? c[u] : kHotRow | h[u];
                F.lrow[at] = (uint16_t)l[u];
                F.out_perm[at] = p[u];
                if (F.src) {
                    F.src[lo + y0 + u * 64 + lane] = at;
                    F.dst[lo + y0 + u * 64 + lane] = F.by_pos ? e[u] : p[u];
                }
            }
        }
    }
    if (lane == 0 && adjacent)
        atomicAdd(&F.C->adjacent, adjacent);
}

// The segments of the other rows, queue by queue in their order: flag[i] for the i-th of queue 0, 1, ...  None of
// them may be a part of a row, or of `must` entries and more.
__global__ void rest_flags_k(const Seg *__restrict__ segs, uint32_t nseg, const uint8_t *__restrict__ row_in,
                             uint32_t must, uint32_t *flag, Seg *__restrict__ out, HubCounters *C)
{
    const uint32_t per_queue = nseg / kSlices, q = blockIdx.y;
    uint32_t mine = 0;
    bool left = false;
    for (uint32_t i = blockIdx.x * kTB + threadIdx.x; i < per_queue; i += gridDim.x * kTB) {
        const uint32_t s = (i / kChunk * kSlices + q) * kChunk + i % kChunk;
        const Seg g = segs[s];
        const bool rest = g.len && !row_in[g.row];
        flag[q * per_queue + i] = rest;
        out[s] = Seg{0, 0, 0, kWholeRow};
        mine += rest;
        left |= rest && (g.slot != kWholeRow || g.len >= must);
    }
    mine = block_sum(mine);
    if (threadIdx.x == 0 && mine)
        atomicAdd(&C->rest[q], mine);
    if (__syncthreads_or(left) && threadIdx.x == 0)
        atomicOr(&C->left_out, 1u);
}
__global__ void rest_segs_k(const Seg *__restrict__ segs, uint32_t nseg, const uint32_t *__restrict__ flag,
                            const uint32_t *__restrict__ at, Seg *__restrict__ out)
{
    const uint32_t per_queue = nseg / kSlices, q = blockIdx.y;
    for (uint32_t i = blockIdx.x * kTB + threadIdx.x; i < per_queue; i += gridDim.x * kTB) {
        if (!flag[q * per_queue + i])
            continue;
        const uint32_t j = at[q * per_queue + i] - at[q * per_queue];
        out[(j / kChunk * kSlices + q) * kChunk + j % kChunk] = segs[(i / kChunk * kSlices + q) * kChunk + i % kChunk];
    }
}

int build_hub_tiles(const DevStream &st, const HubSource &in, HubTiles &out, std::string &err)
{
    out = HubTiles();
    const uint32_t R = in.rows_per_tile, P = in.per_launch, nrows = in.nrows, ncols = in.ncols;
    const uint64_t nnz = in.nnz, nplaces = (uint64_t)P * R;
    if (nnz == 0 || R == 0 || R > kTileMaxRows || P == 0 || in.nseg % (kSlices * kChunk) ||
        (uint64_t)ncols * 1024 + nnz >= (1ull << 32) || in.block_bytes < in.row_bytes)
        return SPC3D_OK;
    // From here to the entries the device waits for launches more than it works, so there are few of them.
    Arena arena(st);
    HIP_OK(arena.reserve(((size_t)nrows + 1) * 9 + ((size_t)ncols + 1) * 12 + (size_t)in.nseg * 8 + nplaces * 16 +
                         (size_t)nnz * 4 + ((size_t)8 << 20)));
    Temp tmp(arena);
    const uint32_t cut = (uint32_t)std::max<uint64_t>(64, nnz / ((uint64_t)P * kTileParts));
    SBuf<uint32_t> sums, before;
    SBuf<uint16_t> block, hot;
    SBuf<uint8_t> row_in;
    SBuf<HubCounters> dC;
    SBuf<TilePlace> place;
    DBuf<uint32_t> tile_rows, slot, col, perm, src, dst, ptr;
    DBuf<uint16_t> lrow;
    DBuf<SplitRow> splits;
    DBuf<Seg> rest;
    const size_t nsums = (size_t)ncols + nrows + 2;
    HIP_OK(sums.alloc(arena, nsums));
    HIP_OK(before.alloc(arena, nsums));
    HIP_OK(row_in.alloc(arena, nrows));
    HIP_OK(block.alloc(arena, ncols));
    HIP_OK(dC.alloc(arena, 1));
    HIP_OK(place.alloc(arena, nplaces));
    HIP_OK(tile_rows.alloc(st, nplaces));
    HIP_OK(slot.alloc(st, nplaces));
    LAUNCH(hub_start_k, std::max<uint64_t>(nsums, nplaces), in.coldeg, (uint64_t)ncols, in.rowptr, (uint64_t)nrows,
           std::max(1u, in.min_row), cut, nplaces, sums.p, row_in.p, tile_rows.p, place.p, dC.p);
    TRY(exclusive_sum(tmp, sums.p, before.p, nsums, st, err));
    const uint32_t *first = before.p + ncols + 1; // of every row its first piece, from total_weight on
    uint32_t upto = 0, total_weight = 0;
    TRY(fetch_all(st, {{&upto, first + nrows, sizeof upto}, {&total_weight, before.p + ncols, sizeof total_weight}},
                  err));
    const uint32_t npc = upto - total_weight;
    // Blocks of columns by number (hot and cold ones mixed: gathers that hit and gathers that miss overlap)
    // whose dense rows take block_bytes of every L2.
    const uint32_t per_block = (uint32_t)std::min<uint64_t>(0xFFFFFFFFull, in.block_bytes / in.row_bytes * 1024);
    const uint32_t nb = total_weight / per_block + 1;
    if (npc == 0 || nb < in.min_blocks || nb > std::min(kFillBlocks, in.max_blocks))
        return SPC3D_OK;
    const bool results = in.results && nb >= in.min_blocks_results;
    if (!results && !in.sums)
        return SPC3D_OK;
    if (in.nhot)
        HIP_OK(hot.alloc(arena, ncols));
    LAUNCH(hub_blocks_k, ncols, before.p, (uint64_t)ncols, per_block, nb, block.p, in.nhot ? hot.p : nullptr);
    if (in.nhot)
        LAUNCH(hot_ranks_k, in.nhot, in.hot_cols, (uint64_t)in.nhot, hot.p);
    // ---- places ----
    HIP_OK(arena.reserve((size_t)npc * 20 + ((size_t)4 << 20)));
    SBuf<uint32_t> key, row_of, id, key_sorted, order, off, tile_n, tptr;
    HIP_OK(key.alloc(arena, npc));
    HIP_OK(row_of.alloc(arena, npc));
    HIP_OK(id.alloc(arena, npc));
    HIP_OK(key_sorted.alloc(arena, npc));
    HIP_OK(order.alloc(arena, npc));
    HIP_OK(off.alloc(arena, nplaces));
    HIP_OK(tile_n.alloc(arena, (size_t)P + 1));
    HIP_OK(tptr.alloc(arena, (size_t)P + 1));
    // cut rows have more than `cut` entries each
    out.split_cap = nnz / cut + 1;
    HIP_OK(splits.alloc(st, out.split_cap));
    LAUNCH(hub_pieces_k, nrows, in.rowptr, (uint64_t)nrows, first, total_weight, key.p, id.p, row_of.p);
    TRY(sort_pairs<uint32_t>(tmp, key.p, key_sorted.p, id.p, order.p, npc, 8, true, st, err));
    LAUNCH(hub_places_k, npc, order.p, row_of.p, (uint64_t)npc, in.rowptr, first, total_weight, P, R,
           place.p, tile_rows.p, slot.p, row_in.p, splits.p, dC.p);
    hipLaunchKernelGGL(hub_offsets_k, dim3(P), dim3(kTileMaxRows), 0, st, place.p, R, off.p, tile_n.p);
    TRY(exclusive_sum(tmp, tile_n.p, tptr.p, (size_t)P + 1, st, err));
    // ---- the other rows' segments ----
    SBuf<uint32_t> flag, at;
    HIP_OK(flag.alloc(arena, in.nseg));
    HIP_OK(at.alloc(arena, in.nseg));
    HIP_OK(rest.alloc(st, in.nseg));
    const dim3 seg_grid((in.nseg / kSlices + kTB * 4 - 1) / (kTB * 4), kSlices);
    hipLaunchKernelGGL(rest_flags_k, seg_grid, dim3(kTB), 0, st, in.segs, in.nseg, row_in.p, in.must, flag.p, rest.p,
                       dC.p);
    TRY(exclusive_sum(tmp, flag.p, at.p, in.nseg, st, err));
    hipLaunchKernelGGL(rest_segs_k, seg_grid, dim3(kTB), 0, st, in.segs, in.nseg, flag.p, at.p, rest.p);
    // ---- entries (room for all: how many are in the tiles is known when they are) ----
    HIP_OK(col.alloc(st, nnz));
    HIP_OK(perm.alloc(st, nnz));
    if (results) {
        HIP_OK(src.alloc(st, nnz));
        HIP_OK(dst.alloc(st, nnz));
    }
    HIP_OK(lrow.alloc(st, nnz));
    HIP_OK(ptr.alloc(st, (size_t)P * nb + 1));
    SBuf<uint32_t> where;
    HIP_OK(where.alloc(arena, nnz));
    const HubFill F = {in.col, in.pos, block.p, in.nhot ? hot.p : nullptr, place.p, off.p, tptr.p, R, nb, in.by_pos,
                       where.p, ptr.p, col.p, perm.p, src.p, dst.p, lrow.p, dC.p};
    hipLaunchKernelGGL(hub_fill_k, dim3(P), dim3(kFillTB), 0, st, F);
    uint32_t n = 0;
    HubCounters hC;
    TRY(fetch_all(st, {{&n, tptr.p + P, sizeof n}, {&hC, dC.p, sizeof hC}}, err));
    if ((uint64_t)n * 2 < nnz || hC.left_out) // (little gained; or the rest is not of short rows alone)
        return SPC3D_OK;
    uint32_t chunks = 0;
    for (uint32_t q = 0; q < kSlices; ++q)
        chunks = std::max(chunks, (hC.rest[q] + kChunk - 1) / kChunk);
    // Results whose neighbours in the tile are mostly their neighbours in the caller's order go straight there:
    // pieces of lines that the same workgroup completes a few blocks later.  (R-MAT 20, rows and columns sorted,
    // three in four, fp64 / fp32 705 -> 685 us and 363 -> 357; a block of R-MAT 24, one in six, 491 -> 546.)
    out.direct = results && !in.pos && (uint64_t)hC.adjacent * 5 >= (uint64_t)n * 3;
    if (out.direct) {
        src.reset();
        dst.reset();
    }
    out.col = col.release();
    out.perm = perm.release();
    out.src = src.release();
    out.dst = dst.release();
    out.lrow = lrow.release();
    out.ptr = ptr.release();
    out.tile_rows = tile_rows.release();
    out.slot = slot.release();
    out.splits = splits.release();
    out.rest = rest.release();
    out.n = n;
    out.ntiles = P;
    out.nblocks = nb;
    out.nsplit = hC.nsplit;
    out.nslots = hC.nslots;
    out.nrest = chunks * kSlices * kChunk;
    return SPC3D_OK;
}

// ii[perm[k]], jj[perm[k]] = row and column of sweep entry k: its tile by bisection over the
// tiles' first bounds, its row from the tile's row list.
__global__ void sweep_coords_k(const uint32_t *__restrict__ ptr, uint32_t ntiles, uint32_t nb,
                               const uint32_t *__restrict__ tile_rows, uint32_t R,
                               const uint16_t *__restrict__ lrow, const uint32_t *__restrict__ col,
                               const uint32_t *__restrict__ perm, uint64_t n, uint32_t *ii,
                               uint32_t *jj)
{
    GRID_STRIDE(k, n)
    {
        uint32_t lo = 0, hi = ntiles; // ptr[lo * nb] <= k < ptr[hi * nb]
        while (hi - lo > 1) {
            const uint32_t mid = lo + (hi - lo) / 2;
            if (ptr[(uint64_t)mid * nb] <= k)
                lo = mid;
            else
                hi = mid;
        }
        const uint32_t at = perm[k];
        ii[at] = tile_rows[(uint64_t)lo * R + lrow[k]];
        jj[at] = col[k];
    }
}

// The same for the entries of a plan in segments (perm null: kernel order is the caller's).
__global__ void seg_coords_k(const Seg *__restrict__ segs, uint64_t nseg,
                             const uint32_t *__restrict__ col, const uint32_t *__restrict__ perm,
                             uint32_t *ii, uint32_t *jj)
{
    GRID_STRIDE(sg, nseg)
    {
        const Seg g = segs[sg];
        for (uint32_t q = g.start; q < g.start + g.len; ++q) {
            const uint32_t at = perm ? perm[q] : q;
            ii[at] = g.row;
            jj[at] = col[q];
        }
    }
}

int sweep_coords_device(const DevStream &st, const SweepPlan &sw, uint32_t *d_ii, uint32_t *d_jj,
                        std::string &err)
{
    if (sw.n == 0)
        return SPC3D_OK;
    LAUNCH(sweep_coords_k, sw.n, sw.ptr, sw.ntiles, sw.nblocks, sw.tile_rows, sw.rows_per_tile,
           sw.lrow, sw.col, sw.perm, sw.n, d_ii, d_jj);
    HIP_OK(hipGetLastError());
    return SPC3D_OK;
}

int seg_coords_device(const DevStream &st, const Seg *d_segs, uint64_t nseg, const uint32_t *d_col,
                      const uint32_t *d_perm, uint32_t *d_ii, uint32_t *d_jj, std::string &err)
{
    if (nseg == 0)
        return SPC3D_OK;
    LAUNCH(seg_coords_k, nseg, d_segs, nseg, d_col, d_perm, d_ii, d_jj);
    HIP_OK(hipGetLastError());
    return SPC3D_OK;
}

int count_adjacent_device(const DevStream &st, const uint32_t *d, uint64_t n, uint64_t *out,
                          std::string &err)
{
    *out = 0;
    if (n < 2)
        return SPC3D_OK;
    DBuf<unsigned long long> acc;
    HIP_OK(acc.alloc(st, 1));
    HIP_OK(hipMemsetAsync(acc.p, 0, sizeof(unsigned long long), st));
    LAUNCH_SMALL(adjacent_k, n, d, n, acc.p);
    unsigned long long seen = 0;
    TRY(fetch(st, &seen, acc.p, sizeof seen, err));
    *out = seen;
    return SPC3D_OK;
}

int inverse_offsets_device(const DevStream &st, const uint32_t *d_perm, uint64_t n, uint32_t base,
                           uint32_t *d_out, std::string &err)
{
    if (n == 0)
        return SPC3D_OK;
    LAUNCH(inverse_offsets_k, n, d_perm, n, base, d_out);
    HIP_OK(hipGetLastError());
    return SPC3D_OK;
}

int gather_u32_device(const DevStream &st, const uint32_t *d_in, const uint32_t *d_idx, uint64_t n,
                      uint32_t *d_out, std::string &err)
{
    if (n == 0)
        return SPC3D_OK;
    LAUNCH(gather_u32_k, n, d_in, d_idx, n, d_out);
    HIP_OK(hipGetLastError());
    return SPC3D_OK;
}

} // namespace spc3d
