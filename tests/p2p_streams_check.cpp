// The rule on what a point-to-point step leaves in the caches goes by the step's bytes, not by its
// pairs: many small pairs, a chunk or two each, do not make a large step.
#include "runtime/batched_p2p.h"

#include <cstdio>
#include <random>

using namespace gpumpi;

int main() {
    std::mt19937_64 rng(7);
    for (int64_t n : {1ll, 64ll, 1000ll, 20000ll, 65536ll, 1000000ll})
        for (uint64_t mib : {1ull, 15ull, 64ull, 256ull, 480ull, 544ull, 1024ull, 4096ull}) {
            uint64_t chunks = 0;
            const uint64_t each = (mib << 20) / (uint64_t)n;
            for (int64_t i = 0; i < n; i++) {
                const uint64_t d = rng() % (1ull << 40), b = each ? each / 2 + rng() % each : 0;
                chunks += b ? ((d + b - 1) >> kP2pChunkShift) - (d >> kP2pChunkShift) + 1 : 0;
            }
            const uint64_t bytes = mib << 20;
            const int want = bytes >= kP2pStores ? kP2pKeepNothing : bytes >= kP2pLoads ? kP2pKeepStores : kP2pCached;
            if (n >= 1000 ? p2p_caching(chunks, n) != want : mib < 32 && p2p_caching(chunks, n) != kP2pCached) {
                std::printf("%lld pairs, %llu MiB: %d\n", (long long)n, (unsigned long long)mib, (int)p2p_caching(chunks, n));
                return 1;
            }
        }
    return 0;
}
