// The work items of the split sort's parts, over part sizes up to the largest that the local
// sort accepts: the items' pieces must follow each other and cover the part.
#include "runtime/bucket.h"

#include <cstdio>

using namespace gpumpi;

static int check(uint32_t c, uint32_t chunk) {
    const uint32_t most = 2 * chunk, items = sort_items(c, most, chunk);
    if (c <= most) return items != (c ? 1u : 0u);
    uint64_t at = 0;
    for (uint32_t k = 0; k < items; k++) {
        const uint32_t i0 = k * chunk;
        if (i0 != at) return 1;
        const uint32_t i1 = sort_item_end(i0, c, chunk);
        if (i1 <= i0 || i1 - i0 > chunk) return 1;
        at = i1;
    }
    return at != c;
}

int main() {
    int bad = 0;
    for (uint32_t chunk : {16384u, 32768u, 49152u, 262144u}) {
        uint32_t sizes[] = {0u, 1u, chunk, 2 * chunk, 2 * chunk + 1, 3 * chunk - 1, 3 * chunk, 3 * chunk + 1, 0x7FFFFFFFu, 0x80000000u,
                            ~0u - 2 * chunk, ~0u - chunk - 1, ~0u - chunk, ~0u - chunk + 1, ~0u - chunk + 2, ~0u - 8191u, ~0u - 8u, ~0u - 1, ~0u};
        for (uint32_t c : sizes)
            if (check(c, chunk)) {
                std::printf("chunk %u: a part of %u keys is not covered\n", chunk, c);
                bad = 1;
            }
    }
    return bad;
}
