// The bucket plan's workgroups: every tile of every rank is one workgroup's, and the XCDs (which
// get the workgroups in turn) share them evenly, however few ranks there are.  The tilings cover
// every rank's keys, and their tables stay within 32 MiB or an eighth of the keys.
#include "runtime/bucket_plan.h"

#include <cstdio>
#include <vector>

using namespace gpumpi;

static int check_tiling(int P, int64_t n, int nb, bool least) {
    const BucketTiling t = bucket_tiling(P, n, nb, least);
    const int64_t per = (int64_t)t.base * t.subs;
    const uint64_t keys = 4 * (uint64_t)P * (uint64_t)n, table = 4 * t.table_words(P, nb);
    const uint64_t most = least ? (n <= 1ll << 30 ? 0 : keys / 8) : keys / 8 > kBucketTableBytes ? keys / 8 : kBucketTableBytes;
    const bool ok = t.subs >= 1 && t.tiles >= 1 && per <= 1ll << 30 && per * t.tiles >= n && per * (t.tiles - 1) < n &&
                    table <= most && (int64_t)P * t.tiles <= 0x7FFFFFF8;
    if (!ok)
        std::printf("P %d n %lld nb %d least %d: base %u subs %u tiles %u, table %llu of %llu bytes\n", P, (long long)n, nb, least,
                    t.base, t.subs, t.tiles, (unsigned long long)table, (unsigned long long)most);
    return ok ? 0 : 1;
}

int main() {
    for (int P : {1, 3, 64, 512, 1100, 65535})
        for (int64_t n : {1ll, 2047ll, 2048ll, 2049ll, 8193ll, 16385ll, 100003ll, 1ll << 18, 6000000ll, 1ll << 27, (1ll << 31) - 1, 1ll << 33})
            for (int nb : {2, 512, 1024, 2048, 4096})
                for (bool least : {false, true})
                    if (check_tiling(P, n, nb, least)) return 1;
    // the tilings of up to 1024 buckets take one tile per workgroup at the usual sizes
    for (int P : {4, 64, 512})
        for (int64_t n : {1024ll, 16384ll, 100003ll, 1ll << 18})
            if (bucket_tiling(P, n, 1024, false).subs != 1) {
                std::printf("P %d n %lld: more than a tile per workgroup\n", P, (long long)n);
                return 1;
            }
    for (int P : {1, 2, 3, 4, 7, 8, 9, 16, 63, 64, 65, 513})
        for (uint32_t tiles : {1u, 2u, 3u, 8u, 17u, 100u}) {
            const uint32_t all = (uint32_t)P * tiles, grid = (all + 7) / 8 * 8;
            std::vector<int> seen(all, 0);
            uint32_t work[8] = {};
            for (uint32_t g = 0; g < grid; g++) {
                int r;
                uint32_t t;
                if (!bucket_tile_of(g, P, tiles, &r, &t)) continue;
                if (r < 0 || r >= P || t >= tiles || seen[(uint32_t)r * tiles + t]++) {
                    std::printf("P %d tiles %u: workgroup %u has rank %d tile %u\n", P, tiles, g, r, t);
                    return 1;
                }
                work[g & 7]++;
            }
            for (uint32_t i = 0; i < all; i++)
                if (!seen[i]) {
                    std::printf("P %d tiles %u: tile %u is no workgroup's\n", P, tiles, i);
                    return 1;
                }
            for (uint32_t x : work)
                if (x > (all + 7) / 8) {
                    std::printf("P %d tiles %u: an XCD has %u of %u tiles\n", P, tiles, x, all);
                    return 1;
                }
        }
    return 0;
}
