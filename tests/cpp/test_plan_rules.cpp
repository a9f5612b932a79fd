// Host-only test of the rules in spcomm3d_amd/csrc/plan_host.h that decide by size.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../spcomm3d_amd/csrc/plan_host.h"

using namespace spc3d;

static int g_fail = 0;
#define CHECK(cond)                                                                               \
    do {                                                                                          \
        if (!(cond)) {                                                                            \
            std::printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond);                           \
            ++g_fail;                                                                             \
        }                                                                                         \
    } while (0)

// The positions that SDDMM over a tile's entries [lo, hi) steps through, as the kernel does in 32
// bits (sweep_sddmm_kernel): `groups` lane groups, batches of 16, the next batch asked for ahead.
// True: every entry is taken once, nothing else is, and no position begins again at 0.
static bool walk(uint32_t lo, uint32_t hi, uint32_t groups)
{
    const uint32_t ub = 16, step = groups * ub, rounds = (hi - lo + step - 1) / step;
    std::vector<uint8_t> taken(hi - lo);
    bool ok = true;
    auto fetch = [&](uint32_t q) { // its length; from a position inside the tile only
        if (q >= hi)
            return 0u;
        ok = ok && q >= lo;
        return hi - q < ub ? hi - q : ub;
    };
    for (uint32_t g = 0; g < groups; ++g) {
        uint32_t p = lo + g * ub, cur = fetch(p);
        for (uint32_t r = 0; r < rounds; ++r, p += step) {
            if (p >= hi)
                continue;
            const uint32_t nxt = fetch(p + step);
            for (uint32_t u = 0; u < cur; ++u) {
                if (p < lo || p + u >= hi)
                    return false;
                ++taken[p + u - lo];
            }
            cur = nxt;
        }
    }
    for (uint8_t n : taken)
        ok = ok && n == 1;
    return ok;
}

static void row_tiles_near_the_end_of_32_bits()
{
    uint64_t most = (1ull << 32) - 1; // the largest pattern that gets tiles
    while (!sweep_fits(most))
        --most;
    CHECK(most == (1ull << 32) - kSweepRound && sweep_fits(0));
    for (uint32_t groups : {16u, 32u, 64u}) // dense rows of 64, 32 and 16 lanes
        for (uint32_t len = 1; len <= 2 * kSweepRound + 1; ++len)
            CHECK(walk((uint32_t)(most - len), (uint32_t)most, groups));
    // (the check sees what it is for: two rounds further the walk goes wrong)
    CHECK(!walk(0xFFFFFFFFu - 100, 0xFFFFFFFFu, 64));
}

// The parts of a bucket cover its ids, each of them once and none past its end, as bucket_count_k takes them, in a
// pattern of n entries that all lie in that bucket or in all of them alike.
static void counts_near_the_end_of_32_bits()
{
    const uint32_t most_entries = 0xFFFFFFFFu;
    for (uint32_t n : {1u, 65535u, 65536u, 65537u, 1u << 22, (1u << 22) + 1, 4228000000u, 4230000000u, most_entries - 63,
                       most_entries - 1, most_entries})
        for (uint32_t nbins : {1u, 2u, 1u << 14, (1u << 14) + 1, 1u << 22, (1u << 22) + 1, 1u << 26}) {
            const CountSizes s = count_sizes(n, nbins);
            CHECK(s.low <= kCountBits && ((uint64_t)s.nbuckets << s.low) >= nbins);
            const uint32_t g = parts_of(n, s.part); // all in one bucket
            CHECK(g >= 1 && g <= s.most);
            CHECK((uint64_t)(g - 1) * s.part < n && (uint64_t)g * s.part >= n);
            CHECK((uint64_t)(g - 1) * s.part <= most_entries); // where the last one begins
            const uint32_t each = n / s.nbuckets, extra = n % s.nbuckets; // all alike
            const uint64_t all = (uint64_t)extra * parts_of(each + 1, s.part) +
                                 (uint64_t)(s.nbuckets - extra) * parts_of(each, s.part);
            CHECK(all <= s.most);
        }
    CHECK(parts_of(0, 1 << 16) == 0);
}

int main()
{
    counts_near_the_end_of_32_bits();
    row_tiles_near_the_end_of_32_bits();
    std::printf(g_fail ? "%d checks FAILED\n" : "PASSED\n", g_fail);
    return g_fail != 0;
}
