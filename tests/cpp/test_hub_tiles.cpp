// build_hub_tiles (spcomm3d_amd/csrc/plan_device.hip) on small patterns, at the edges that a plan reaches only with many
// millions of entries: tiles without rows, no cut row and nothing but cut rows, rows that just miss a place, few and
// as many blocks of columns as there may be, duplicates, hot columns, results by the caller's position and by the
// source's, patterns that get no tiles.  Every array against one made here from the description in plan_device.h.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdio>
#include <numeric>
#include <random>
#include <string>
#include <vector>

#include "../../spcomm3d_amd/csrc/plan_device.h"

using namespace spc3d;
using std::vector;
typedef uint32_t u32;

static int g_fail = 0;
static std::string g_case;
#define CHECK(cond)                                                                               \
    do {                                                                                          \
        if (!(cond)) {                                                                            \
            std::printf("FAIL %s:%d: %s (%s)\n", __FILE__, __LINE__, #cond, g_case.c_str());      \
            ++g_fail;                                                                             \
        }                                                                                         \
    } while (0)

struct Pattern {
    vector<u32> rowptr{0}, col, deg;
    vector<Seg> segs; // a row's, in queues
    u32 nrows() const { return (u32)rowptr.size() - 1; }
};

// Rows of the given lengths; segments of at most seg_max entries, dealt to the queues row by row.
static Pattern make(const vector<u32> &lengths, u32 ncols, u32 seg_max, u32 distinct_cols, unsigned seed)
{
    Pattern p;
    std::mt19937 rng(seed);
    p.deg.assign(ncols, 0);
    vector<vector<Seg>> queue(kSlices);
    for (u32 r = 0; r < lengths.size(); ++r) {
        for (u32 i = 0; i < lengths[r]; ++i) {
            // (skewed, and every column of `distinct_cols` at least now and then)
            const u32 c = i % 4 ? (u32)((uint64_t)rng() * rng() >> 32) % distinct_cols : (u32)(rng() % distinct_cols);
            p.col.push_back(c);
            ++p.deg[c];
        }
        const u32 at = p.rowptr.back(), parts = (lengths[r] + seg_max - 1) / seg_max;
        p.rowptr.push_back(at + lengths[r]);
        for (u32 k = 0; k < parts; ++k)
            queue[r % kSlices].push_back(
                Seg{r, at + k * seg_max, std::min(seg_max, lengths[r] - k * seg_max), parts > 1 ? k : kWholeRow});
    }
    size_t most = 1;
    for (auto &q : queue)
        most = std::max(most, q.size());
    const size_t chunks = (most + kChunk - 1) / kChunk;
    p.segs.assign(chunks * kChunk * kSlices, Seg{0, 0, 0, kWholeRow});
    for (u32 q = 0; q < kSlices; ++q)
        for (size_t j = 0; j < queue[q].size(); ++j)
            p.segs[(j / kChunk * kSlices + q) * kChunk + j % kChunk] = queue[q][j];
    return p;
}

struct Want {
    u32 nblocks = 0, nslots = 0, nrest = 0;
    uint64_t n = 0;
    bool none = false;
    vector<u32> col, perm, ptr, tile_rows, slot, src, dst;
    vector<uint16_t> lrow;
    vector<SplitRow> splits;
    vector<Seg> rest;
};

static Want model(const Pattern &p, const HubSource &in, const vector<u32> &pos, const vector<u32> &hot)
{
    Want w;
    const u32 R = in.rows_per_tile, P = in.per_launch, nrows = p.nrows();
    const u32 cut = (u32)std::max<uint64_t>(64, in.nnz / ((uint64_t)P * kTileParts));
    // blocks of columns
    vector<u32> block(in.ncols);
    u32 sum = 0;
    const u32 per_block = (u32)(in.block_bytes / in.row_bytes * 1024);
    for (u32 c = 0; c < in.ncols; ++c) {
        block[c] = sum / per_block;
        u32 miss = 1024;
        for (u32 k = 0; k < std::min(p.deg[c], 52u); ++k)
            miss = miss * 7 / 8;
        sum += 1024 - miss;
    }
    w.nblocks = sum / per_block + 1;
    for (u32 &b : block)
        b = std::min(b, w.nblocks - 1);
    // pieces, longest first to an eighth of an octave
    struct Piece {
        u32 key, row, i, np;
    };
    vector<Piece> pieces;
    for (u32 r = 0; r < nrows; ++r) {
        const u32 len = p.rowptr[r + 1] - p.rowptr[r];
        if (len < std::max(1u, in.min_row))
            continue;
        const u32 np = (len + cut - 1) / cut, each = len / np;
        u32 e = 0;
        while (each >> (e + 1))
            ++e;
        for (u32 i = 0; i < np; ++i)
            pieces.push_back({e * 8 + (u32)(((uint64_t)each << 3 >> e) & 7), r, i, np});
    }
    if (pieces.empty() || w.nblocks < in.min_blocks || w.nblocks > in.max_blocks) {
        w.none = true;
        return w;
    }
    std::stable_sort(pieces.begin(), pieces.end(), [](const Piece &a, const Piece &b) { return a.key > b.key; });
    w.tile_rows.assign((size_t)P * R, 0xFFFFFFFFu);
    w.slot.assign((size_t)P * R, 0);
    vector<vector<u32>> entries((size_t)P * R); // of the source
    vector<char> row_in(nrows, 0);
    for (u32 j = 0; j < pieces.size(); ++j) {
        const Piece &q = pieces[j];
        if ((uint64_t)(j - q.i) + q.np > (uint64_t)P * R)
            continue;
        const u32 l = j / P, x = j % P;
        const size_t at = (size_t)(l & 1 ? P - 1 - x : x) * R + l;
        w.tile_rows[at] = q.row;
        w.slot[at] = q.np > 1 ? j : kWholeRow;
        row_in[q.row] = 1;
        const u32 lo = p.rowptr[q.row], hi = p.rowptr[q.row + 1];
        for (u32 g = q.i; lo + g * kTileGroup < hi; g += q.np)
            for (u32 e = lo + g * kTileGroup; e < std::min(hi, lo + (g + 1) * kTileGroup); ++e)
                entries[at].push_back(e);
        if (q.np > 1 && q.i == 0) {
            w.splits.push_back(SplitRow{q.row, j, q.np, 0});
            w.nslots = std::max(w.nslots, j + q.np);
        }
    }
    // entries
    for (u32 t = 0; t < P; ++t) {
        struct E {
            u32 block, place, at, h;
        };
        vector<E> es;
        u32 h = (u32)w.n;
        for (u32 l = 0; l < R; ++l)
            for (u32 e : entries[(size_t)t * R + l])
                es.push_back({block[p.col[e]], l, e, h++});
        std::stable_sort(es.begin(), es.end(), [](const E &a, const E &b) { return a.block < b.block; });
        for (u32 b = 0, k = 0; b < w.nblocks; ++b) {
            while (k < es.size() && es[k].block < b)
                ++k;
            w.ptr.push_back((u32)w.n + k);
        }
        w.src.resize(w.n + es.size());
        w.dst.resize(w.n + es.size());
        for (const E &e : es) {
            const auto hit = std::find(hot.begin(), hot.end(), p.col[e.at]);
            w.col.push_back(hit == hot.end() ? p.col[e.at] : kHotRow | (u32)(hit - hot.begin()));
            w.perm.push_back(e.at);
            w.lrow.push_back((uint16_t)e.place);
            w.src[e.h] = (u32)w.perm.size() - 1;
            w.dst[e.h] = in.by_pos && !pos.empty() ? pos[e.at] : e.at;
        }
        w.n += es.size();
    }
    w.ptr.push_back((u32)w.n);
    // the other rows
    bool left_out = false;
    size_t most = 0;
    vector<vector<Seg>> rest(kSlices);
    for (u32 q = 0; q < kSlices; ++q) {
        for (size_t i = 0; i < p.segs.size() / kSlices; ++i) {
            const Seg &s = p.segs[(i / kChunk * kSlices + q) * kChunk + i % kChunk];
            if (!s.len || row_in[s.row])
                continue;
            left_out |= s.slot != kWholeRow || s.len >= in.must;
            rest[q].push_back(s);
        }
        most = std::max(most, rest[q].size());
    }
    w.nrest = (u32)((most + kChunk - 1) / kChunk * kSlices * kChunk);
    w.rest.assign(w.nrest, Seg{0, 0, 0, kWholeRow});
    for (u32 q = 0; q < kSlices; ++q)
        for (size_t j = 0; j < rest[q].size(); ++j)
            w.rest[(j / kChunk * kSlices + q) * kChunk + j % kChunk] = rest[q][j];
    w.none = w.n * 2 < in.nnz || left_out;
    return w;
}

static DevPool g_pool;
static bool g_host = false; // what is expected only, without a device
template <typename T> static T *put(const vector<T> &v)
{
    void *d = nullptr;
    if (v.empty())
        return nullptr;
    if (g_pool.get(&d, v.size() * sizeof(T)) != hipSuccess ||
        hipMemcpy(d, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess) {
        std::printf("no device memory\n");
        std::exit(1);
    }
    return static_cast<T *>(d);
}
template <typename T> static vector<T> take(T *d, size_t n)
{
    vector<T> v(n);
    if (n)
        CHECK(hipMemcpy(v.data(), d, n * sizeof(T), hipMemcpyDeviceToHost) == hipSuccess);
    if (d)
        g_pool.put(d);
    return v;
}
static bool same(const Seg &a, const Seg &b)
{
    return a.row == b.row && a.start == b.start && a.len == b.len && a.slot == b.slot;
}

// tiles: whether the pattern is meant to have them
static void check(const char *name, bool tiles, const Pattern &p, HubSource in, u32 nhot = 0, bool with_pos = false)
{
    g_case = name;
    std::printf("%s\n", name);
    std::fflush(stdout);
    in.nrows = p.nrows();
    in.ncols = (u32)p.deg.size();
    in.nnz = p.col.size();
    vector<u32> pos, hot;
    std::mt19937 rng(7);
    if (with_pos) {
        pos.resize(in.nnz);
        std::iota(pos.begin(), pos.end(), 0u);
        std::shuffle(pos.begin(), pos.end(), rng);
    }
    for (u32 c = in.ncols; hot.size() < nhot;)
        hot.push_back(--c);
    const Want w = model(p, in, pos, hot);
    CHECK(w.none == !tiles);
    if (g_host) {
        std::printf("  %llu of %llu entries in tiles, %u blocks, %zu cut rows, %u other segments\n", (unsigned long long)w.n,
                    (unsigned long long)in.nnz, w.nblocks, w.splits.size(), w.nrest);
        return;
    }
    in.rowptr = put(p.rowptr);
    in.coldeg = put(p.deg);
    in.col = put(p.col);
    in.pos = put(pos);
    in.segs = put(p.segs);
    in.nseg = (u32)p.segs.size();
    in.hot_cols = put(hot);
    in.nhot = nhot;
    HubTiles t;
    std::string err;
    CHECK(build_hub_tiles({nullptr, &g_pool}, in, t, err) == 0);
    CHECK((t.n != 0) == tiles);
    if (t.n && tiles) {
        CHECK(t.n == w.n && t.ntiles == in.per_launch && t.nblocks == w.nblocks);
        CHECK(t.nsplit == w.splits.size() && t.nslots == w.nslots && t.nrest == w.nrest);
        CHECK(w.splits.size() <= t.split_cap);
        CHECK(t.direct ? in.results && !in.pos && !t.src : !t.src == !in.results);
        CHECK(take(t.ptr, (size_t)t.ntiles * t.nblocks + 1) == w.ptr);
        CHECK(take(t.col, t.n) == w.col);
        CHECK(take(t.perm, t.n) == w.perm);
        CHECK(take(t.lrow, t.n) == w.lrow);
        const vector<u32> rows = take(t.tile_rows, w.tile_rows.size()), slot = take(t.slot, w.slot.size());
        CHECK(rows == w.tile_rows);
        for (size_t i = 0; i < rows.size(); ++i)
            if (rows[i] != 0xFFFFFFFFu)
                CHECK(slot[i] == w.slot[i]);
        if (t.src) {
            CHECK(take(t.src, t.n) == w.src);
            CHECK(take(t.dst, t.n) == w.dst);
        }
        vector<SplitRow> splits = take(t.splits, t.nsplit);
        std::sort(splits.begin(), splits.end(), [](auto &a, auto &b) { return a.first_slot < b.first_slot; });
        for (size_t i = 0; i < std::min(splits.size(), w.splits.size()); ++i)
            CHECK(splits[i].row == w.splits[i].row && splits[i].first_slot == w.splits[i].first_slot &&
                  splits[i].nslots == w.splits[i].nslots);
        const vector<Seg> rest = take(t.rest, t.nrest);
        CHECK(rest.size() == w.rest.size() && std::equal(rest.begin(), rest.end(), w.rest.begin(), same));
    }
    for (const void *d : {(const void *)in.rowptr, (const void *)in.coldeg, (const void *)in.col, (const void *)in.pos,
                          (const void *)in.segs, (const void *)in.hot_cols})
        if (d)
            g_pool.put(const_cast<void *>(d));
}

static vector<u32> lengths(size_t n, u32 lo, u32 hi, unsigned seed)
{
    std::mt19937 rng(seed);
    vector<u32> v(n);
    for (u32 &x : v)
        x = lo + rng() % (hi - lo + 1);
    return v;
}

int main(int argc, char **argv)
{
    g_host = argc > 1 && std::string(argv[1]) == "--host";
    int devices = 0;
    if (!g_host && (hipGetDeviceCount(&devices) != hipSuccess || devices == 0)) {
        std::printf("no device\n");
        return 1;
    }
    if (!g_host)
        g_pool.open(0, (size_t)1 << 30);
    HubSource base;
    base.rows_per_tile = 32;
    base.per_launch = 16;
    base.min_row = 8;
    base.must = 128;
    base.row_bytes = 512;
    base.block_bytes = 40 * 512; // about 40 columns that are met often
    base.min_blocks = 1;
    base.max_blocks = 1027;

    const vector<u32> mixed = lengths(700, 0, 60, 1);
    check("no row is cut, short rows beside the tiles", true, make(mixed, 400, 2048, 400, 2), base);
    check("as many columns in one block as there are", true, make(mixed, 30, 2048, 30, 3), base);
    check("rows in fewer tiles than there are", true, make(lengths(5, 40, 60, 4), 100, 2048, 100, 5), base);
    check("one row", true, make({64}, 100, 2048, 100, 6), base);
    check("one row, one entry over the cut", true, make({65}, 100, 2048, 100, 6), base);
    {
        HubSource in = base;
        in.rows_per_tile = 64;
        check("every row is cut", true, make(lengths(20, 3000, 9000, 7), 500, 20000, 500, 8), in);
    }
    {
        vector<u32> v = mixed;
        v[17] = 5000; // of 17 and more groups to a piece, the last of them not full
        v[400] = 65;
        v[401] = 80;
        v[402] = 81;
        check("cut rows among others", true, make(v, 400, 20000, 400, 9), base);
        HubSource in = base;
        in.by_pos = false;
        check("results in the source's order", true, make(v, 400, 20000, 400, 9), in);
        check("results in the source's order, the caller's another", true, make(v, 400, 20000, 400, 9), in, 0, true);
        in.by_pos = true;
        check("results at the caller's positions", true, make(v, 400, 20000, 400, 9), in, 0, true);
        in.results = false;
        check("no results", true, make(v, 400, 20000, 400, 9), in);
        check("hot columns", true, make(v, 400, 20000, 400, 9), base, 37);
        in = base;
        in.min_row = 30;
        check("only longer rows", true, make(v, 400, 20000, 400, 9), in);
    }
    check("the same column again and again", true, make(mixed, 400, 2048, 3, 10), base);
    {
        HubSource in = base; // 48 places
        in.rows_per_tile = 16;
        in.per_launch = 3;
        vector<u32> v(60, 40);
        check("as many rows as places and more", true, make(v, 200, 2048, 200, 11), in);
        v.assign(48, 40);
        check("as many rows as places", true, make(v, 200, 2048, 200, 11), in);
        v.assign(49, 40);
        check("a row more than places", true, make(v, 200, 2048, 200, 11), in);
        v.assign(46, 64);
        v.push_back(127);
        check("a cut row that just has its places", true, make(v, 200, 20000, 200, 12), in);
        v.push_back(64);
        check("a cut row that just misses its places", true, make(v, 200, 20000, 200, 12), in);
        v.back() = 130; // its segment is one that has to be in a tile
        check("a long row left out", false, make(v, 200, 20000, 200, 12), in);
        v.back() = 120;
        check("a row in two segments left out", false, make(v, 200, 100, 200, 12), in);
        v.assign(200, 60);
        check("less than half of the entries", false, make(v, 200, 2048, 200, 13), in);
    }
    for (u32 rows : {512u, 256u, 128u}) {
        HubSource in = base;
        in.rows_per_tile = rows;
        in.per_launch = 256;
        check("places of the kernels", true, make(lengths(3000, 1, 300, rows), 3000, 20000, 3000, rows), in);
    }
    for (u32 blocks : {4u, 64u, 65u, 1027u}) {
        HubSource in = base;
        in.block_bytes = 512;
        in.per_launch = 4;
        in.rows_per_tile = 128;
        // columns of one entry each take an eighth of one, of 60 all of it
        Pattern p = make(lengths(512, 100, 140, blocks), 4 * blocks, 2048, blocks, blocks);
        in.must = 256;
        u32 sum = 0;
        for (u32 d : p.deg) {
            u32 miss = 1024;
            for (u32 k = 0; k < std::min(d, 52u); ++k)
                miss = miss * 7 / 8;
            sum += 1024 - miss;
        }
        const u32 nb = sum / 1024 + 1;
        if (nb <= 1027) {
            in.min_blocks = nb;
            check("blocks of columns", true, p, in);
            in.min_blocks = nb + 1;
            check("a block too few", false, p, in);
            in.min_blocks = 1;
        }
        in.max_blocks = nb - 1;
        check("a block too many", false, p, in);
    }
    check("no row is long enough", false, make(lengths(300, 0, 7, 14), 100, 2048, 100, 15), base);
    if (!g_host)
        g_pool.trim();
    std::printf(g_fail ? "%d checks FAILED\n" : "PASSED\n", g_fail);
    return g_fail != 0;
}
