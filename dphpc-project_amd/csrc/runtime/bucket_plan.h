// The bucket plan's host side: how the keys are cut into workgroups, and the launches.
#pragma once

#include "bucket.h"

namespace gpumpi {

// How the keys are cut: `tiles` workgroups per rank, each `subs` tiles of `base` keys one after
// the other (16 keys per thread; 4 where that leaves less than two workgroups per CU).
// One tile per workgroup while the table of counts (4 B per workgroup and bucket) takes at most
// 32 MiB or an eighth of the keys; 4096 buckets would take half.  With one workgroup per rank
// there is no table, only the ranks' prefixes: `least` asks for that, as far as a workgroup's
// keys can be counted in 32 bits, where memory for more is not to be had.
struct BucketTiling {
    uint32_t threads, base, subs, tiles;
    bool small;
    uint64_t table_words(int P, int nb) const { return tiles > 1 ? (uint64_t)P * tiles * (uint64_t)nb : 0; }
    static uint64_t prefix_words(int P, int nb) { return (uint64_t)P * (uint64_t)(nb + 1); }
};
constexpr uint64_t kBucketTableBytes = 32u << 20;
inline BucketTiling bucket_tiling(int P, int64_t n, int nb, bool least) {
    BucketTiling t;
    t.threads = nb <= 1024 ? 1024 : 512;
    t.small = (int64_t)P * ((n + 16 * t.threads - 1) / (16 * t.threads)) < 512;
    t.base = (t.small ? 4 : 16) * t.threads;
    const uint64_t all = ((uint64_t)n + t.base - 1) / t.base, keys = 4 * (uint64_t)P * (uint64_t)n;
    uint64_t most = (keys / 8 > kBucketTableBytes ? keys / 8 : kBucketTableBytes) / (4 * (uint64_t)nb);   // workgroups
    if (most > 0x7FFFFFF0u) most = 0x7FFFFFF0u;     // a grid's limit
    const uint64_t per_rank = least || most < (uint64_t)P ? 1 : most / (uint64_t)P;
    uint64_t subs = (all + per_rank - 1) / per_rank;
    if (subs > 0x40000000u / t.base) subs = 0x40000000u / t.base;
    t.subs = (uint32_t)subs;
    t.tiles = (uint32_t)((all + subs - 1) / subs);
    return t;
}

// Scratch: the buckets' running totals, the table, the ranks' prefixes.
inline size_t bucket_scratch_bytes(const BucketTiling& t, int P, int nb) {
    return sizeof(int64_t) * (size_t)nb + sizeof(uint32_t) * (BucketTiling::prefix_words(P, nb) + t.table_words(P, nb));
}

static auto bucket_scatter_for(bool narrow, bool small, bool turns) {
    if (turns)
        return narrow ? (small ? &bucket_scatter_kernel<1024, 4, 1024, true> : &bucket_scatter_kernel<1024, 16, 1024, true>)
                      : (small ? &bucket_scatter_kernel<512, 4, 4096, true> : &bucket_scatter_kernel<512, 16, 4096, true>);
    return narrow ? (small ? &bucket_scatter_kernel<1024, 4, 1024, false> : &bucket_scatter_kernel<1024, 16, 1024, false>)
                  : (small ? &bucket_scatter_kernel<512, 4, 4096, false> : &bucket_scatter_kernel<512, 16, 4096, false>);
}

static void bucket_plan_launch(const BucketTiling& t, const uint32_t* keys, int P, int64_t n, int shift, int nb, void* scratch,
                               uint32_t* out, int32_t* scounts, int32_t* sdispls, int32_t* lo, int32_t* hi, hipStream_t s) {
    const bool cols = P > 64;   // up to 64 ranks the splitters' workgroup sums the columns itself
    const uint32_t tiles = t.tiles, grid = ((uint32_t)P * tiles + 7) / 8 * 8;
    int64_t* acc = (int64_t*)scratch;
    uint32_t* tile_cnt = (uint32_t*)(acc + nb);
    uint32_t* prefix = tile_cnt + t.table_words(P, nb);     // no table: tile_cnt == prefix
    hipLaunchKernelGGL(bucket_tile_hist_kernel, dim3(grid), dim3(kBucketThreads), sizeof(uint32_t) * nb, s, keys, P, n, shift,
                       nb, t.base * t.subs, tiles, tile_cnt, tiles > 1 ? nb : nb + 1);
    hipLaunchKernelGGL(bucket_rank_scan_kernel, dim3(P), dim3(kBucketThreads), 0, s, nb, tiles, tile_cnt, prefix);
    if (cols)
        hipLaunchKernelGGL(bucket_colsum_kernel, dim3((nb + kWave - 1) / kWave), dim3(kBucketThreads), 0, s, prefix, P, nb, acc);
    hipLaunchKernelGGL(bucket_splitters_kernel, dim3(1), dim3(kBucketThreads), 0, s, cols ? acc : nullptr, prefix, P, nb, n, lo,
                       hi);
    hipLaunchKernelGGL(bucket_scatter_for(nb <= 1024, t.small, t.subs > 1), dim3(grid), dim3(t.threads), 0, s, keys, P, n, shift,
                       nb, tiles, t.subs, tile_cnt, prefix, lo, hi, out, scounts, sdispls);
}

}  // namespace gpumpi
