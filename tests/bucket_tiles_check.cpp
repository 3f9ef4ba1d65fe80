// The bucket plan's workgroups: every tile of every rank is one workgroup's, and the XCDs (which
// get the workgroups in turn) share them evenly, however few ranks there are.
#include "runtime/bucket.h"

#include <cstdio>
#include <vector>

using namespace gpumpi;

int main() {
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
