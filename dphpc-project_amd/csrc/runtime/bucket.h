// Device kernels of the bucket-sort caller of the exchange (the NPB IS rank() shape,
// toolchain_tests/npb/NPB3.4.1/NPB3.4-MPI/IS/is.c:631-928) for the batched path:
//   gen_keys      seeded keys: uniform [0, 2^key_bits), Zipf(s) by inverse CDF, or the
//                 NPB IS LCG (randlc/find_my_seed/create_seq, is.c:406-537) evaluated in
//                 exact integer arithmetic with per-thread jump-ahead
//   bucket_*      per-rank bucket histograms, NPB splitters (is.c:721-751: rank j takes
//                 buckets until the global running total reaches (j+1)*n), send counts and
//                 displacements, stable bucketing (is.c:680-688)
//   sort_*        counting sort of the received keys (is.c:785-833, placement as
//                 full_verify is.c:545-560)
#pragma once

#include "philox.h"
#include "common.h"
#include "copy.h"

namespace gpumpi {

constexpr uint64_t kNpbA = 1220703125ull;
constexpr uint64_t kNpbSeed = 314159265ull;
constexpr uint64_t kMask46 = (1ull << 46) - 1;

__host__ __device__ __forceinline__ uint64_t lcg_pow(uint64_t a, uint64_t e) {
    uint64_t r = 1;
    while (e) {
        if (e & 1) r = (r * a) & kMask46;
        a = (a * a) & kMask46;
        e >>= 1;
    }
    return r;
}

// find_my_seed (is.c:470-510): s * (a^(2^mq))^kn mod 2^46 with mq = floor(log2(nn/np)).
__host__ __device__ __forceinline__ uint64_t npb_rank_seed(int kn, int np, int64_t nn) {
    int64_t nq = nn / np;
    int mq = 0;
    for (; nq > 1; mq++, nq /= 2) {}
    uint64_t an = kNpbA;
    for (int i = 0; i < mq; i++) an = (an * an) & kMask46;
    return (kNpbSeed * lcg_pow(an, (uint64_t)kn)) & kMask46;
}

// NPB IS class parameters and partial-verification tables (is.c:57-104, 264-287).
struct NpbClassInfo {
    int total_keys_log2, max_key_log2, num_buckets_log2;
    int64_t test_index[5], test_rank[5];
};

__host__ __device__ inline bool npb_class_info(char cls, NpbClassInfo& c) {
    int64_t ti[5], tr[5];
    switch (cls) {
    case 'S': {
        c.total_keys_log2 = 16; c.max_key_log2 = 11; c.num_buckets_log2 = 9;
        const int64_t a[5] = {48427, 17148, 23627, 62548, 4431}, b[5] = {0, 18, 346, 64917, 65463};
        for (int i = 0; i < 5; i++) { ti[i] = a[i]; tr[i] = b[i]; }
        break;
    }
    case 'W': {
        c.total_keys_log2 = 20; c.max_key_log2 = 16; c.num_buckets_log2 = 10;
        const int64_t a[5] = {357773, 934767, 875723, 898999, 404505},
                      b[5] = {1249, 11698, 1039987, 1043896, 1048018};
        for (int i = 0; i < 5; i++) { ti[i] = a[i]; tr[i] = b[i]; }
        break;
    }
    case 'A': {
        c.total_keys_log2 = 23; c.max_key_log2 = 19; c.num_buckets_log2 = 10;
        const int64_t a[5] = {2112377, 662041, 5336171, 3642833, 4250760},
                      b[5] = {104, 17523, 123928, 8288932, 8388264};
        for (int i = 0; i < 5; i++) { ti[i] = a[i]; tr[i] = b[i]; }
        break;
    }
    case 'B': {
        c.total_keys_log2 = 25; c.max_key_log2 = 21; c.num_buckets_log2 = 10;
        const int64_t a[5] = {41869, 812306, 5102857, 18232239, 26860214},
                      b[5] = {33422937, 10244, 59149, 33135281, 99};
        for (int i = 0; i < 5; i++) { ti[i] = a[i]; tr[i] = b[i]; }
        break;
    }
    case 'C': {
        c.total_keys_log2 = 27; c.max_key_log2 = 23; c.num_buckets_log2 = 10;
        const int64_t a[5] = {44172927, 72999161, 74326391, 129606274, 21736814},
                      b[5] = {61147, 882988, 266290, 133997595, 133525895};
        for (int i = 0; i < 5; i++) { ti[i] = a[i]; tr[i] = b[i]; }
        break;
    }
    default:
        return false;
    }
    for (int i = 0; i < 5; i++) { c.test_index[i] = ti[i]; c.test_rank[i] = tr[i]; }
    return true;
}

// Expected rank of test key i at `iteration` (is.c:849-905).
__host__ __device__ inline int64_t npb_expected_rank(char cls, int i, int iteration, int64_t r) {
    switch (cls) {
    case 'S': return i <= 2 ? r + iteration : r - iteration;
    case 'W': return i < 2 ? r + iteration - 2 : r - iteration;
    case 'A': return i <= 2 ? r + iteration - 1 : r - (iteration - 1);
    case 'B': return (i == 1 || i == 2 || i == 4) ? r + iteration : r - iteration;
    default: return i <= 2 ? r + iteration : r - iteration;  // 'C'
    }
}

// Key i of rank r for the uniform (dist 0) and Zipf (dist 1) workloads.
__host__ __device__ __forceinline__ uint32_t gen_key(int dist, uint64_t seed, int r, uint32_t step,
                                                     int64_t i, int key_bits, const double* cdf,
                                                     int64_t ncdf) {
    if (dist == 0) {
        u32x4v v = rank_stream(seed, r, step, (uint64_t)(i >> 2), kStreamKeys);
        return pick(v, (int)(i & 3)) >> (32 - key_bits);
    }
    u32x4v v = rank_stream(seed, r, step, (uint64_t)(i >> 1), kStreamZipf);
    const int h = 2 * (int)(i & 1);
    const double u = unit53(pick(v, h), pick(v, h + 1));
    int64_t lo = 0, hi = ncdf - 1;
    while (lo < hi) {
        int64_t mid = lo + (hi - lo) / 2;
        if (cdf[mid] > u) hi = mid; else lo = mid + 1;
    }
    return (uint32_t)lo;
}

// NPB IS create_seq key i of rank r: (x1+x2+x3+x4) >> (48 - max_key_log2), where the x's
// are the next four LCG states of the rank's sequence (which starts at the rank seed).
__host__ __device__ __forceinline__ uint32_t npb_key(int r, int P, int64_t total, int64_t i,
                                                     int max_key_log2) {
    uint64_t x = npb_rank_seed(r, P, 4 * total);
    x = (x * lcg_pow(kNpbA, 4ull * (uint64_t)i)) & kMask46;
    uint64_t s = 0;
    for (int j = 0; j < 4; j++) {
        x = (x * kNpbA) & kMask46;
        s += x;
    }
    return (uint32_t)(s >> (48 - max_key_log2));
}

static __global__ void gen_keys_kernel(uint32_t* keys, int P, int64_t n, uint64_t seed, uint32_t step,
                                int dist, int key_bits, const double* cdf, int64_t ncdf) {
    const int64_t total = (int64_t)P * n;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total;
         g += (int64_t)gridDim.x * blockDim.x) {
        const int r = (int)(g / n);
        const int64_t i = g - (int64_t)r * n;
        keys[g] = dist == 2 ? npb_key(r, P, total, i, key_bits)
                            : gen_key(dist, seed, r, step, i, key_bits, cdf, ncdf);
    }
}

// ------------------------------------------------------------------ bucket plan
// Each rank's keys are cut into tiles of consecutive keys, one or a few per workgroup
// (bucket_plan.h):
//   bucket_tile_hist  the tile's keys per bucket
//   bucket_rank_scan  per rank: exclusive prefix of the tiles' counts within each bucket, and
//                     of the buckets within the rank
//   bucket_colsum     the same prefix summed over the ranks (many ranks only)
//   bucket_splitters  which buckets each rank receives
//   bucket_scatter    the tile's keys to their stable places; the first tile of a rank also
//                     writes the rank's send counts and displacements
// HBM traffic: the keys read twice and written once, plus 4 table passes of 4 B per workgroup
// and bucket.  Measured at 512 ranks x 2^18 keys, 1024 buckets: tile_hist 145-150 us (3.7 TB/s
// read; the LDS atomics bound it, 256 threads per workgroup took 158), rank_scan 16, colsum 11,
// splitters 5, scatter 321 us (3.3 TB/s).  One wavefront per rank, 64
// keys per step (the former scatter), was a serial chain of n / 64 steps on P waves: 5676 us
// there and 208 us at 4 ranks x 2^14, now 8.5; the column sums by one thread per bucket 139 us.
constexpr int kBucketThreads = 1024;

// Exclusive sum over the workgroup (NT threads, a multiple of 64), and the total.  `part`
// holds one word per wavefront; it is free again after the caller's next barrier.
template <int NT>
__device__ __forceinline__ uint32_t block_excl_sum(uint32_t v, uint32_t* part, uint32_t* total) {
    const int l = lane(), w = threadIdx.x >> 6;
    uint32_t inc = v;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t u = (uint32_t)__shfl_up((int)inc, o);
        if (l >= o) inc += u;
    }
    if (l == kWave - 1) part[w] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int k = 0; k < NT / kWave; k++) {
        const uint32_t x = part[k];
        before += k < w ? x : 0u;
        all += x;
    }
    *total = all;
    return before + inc - v;
}

// Workgroup g of a grid of 8 * ceil(P * tiles / 8): workgroups are dealt to the 8 XCDs in turn,
// so each XCD gets an eighth of all tiles in a row, and its L2 joins the pieces of a 128-byte
// line that neighbouring tiles of a rank write.  (With whole ranks dealt to the XCDs, fewer
// than 8 ranks left XCDs idle: 1 rank x 2^27 keys 3824 us, 1637 so; 4 x 2^22 194 and 114.)  false: no such tile.
__host__ __device__ __forceinline__ bool bucket_tile_of(uint32_t g, int P, uint32_t tiles, int* r, uint32_t* tile) {
    const uint32_t all = (uint32_t)P * tiles, at = (g & 7) * ((all + 7) / 8) + (g >> 3);
    *r = (int)(at / tiles);
    *tile = at % tiles;
    return at < all;
}

// tile_cnt: [P][tiles] rows of nb counts, `stride` words apart, every count written.
static __global__ __launch_bounds__(kBucketThreads) void bucket_tile_hist_kernel(
    const uint32_t* keys, int P, int64_t n, int shift, int nb, uint32_t tile_keys, uint32_t tiles,
    uint32_t* tile_cnt, int stride) {
    extern __shared__ uint32_t lh[];
    int r;
    uint32_t tile;
    if (!bucket_tile_of(blockIdx.x, P, tiles, &r, &tile)) return;
    for (int b = threadIdx.x; b < nb; b += kBucketThreads) lh[b] = 0;
    __syncthreads();
    const int64_t i0 = (int64_t)tile * tile_keys;
    const uint32_t m = (uint32_t)(n - i0 < (int64_t)tile_keys ? n - i0 : (int64_t)tile_keys);
    const uint32_t* k = keys + (int64_t)r * n + i0;
    constexpr int kU = 4;       // 16-byte loads in flight per thread
    uint32_t i0v = 4u * threadIdx.x;
    for (; i0v + 4u * (kU - 1) * kBucketThreads + 4 <= m; i0v += 4u * kU * kBucketThreads) {
        u32x4 v[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) v[u] = gload16((uint64_t)(uintptr_t)(k + i0v + 4u * u * kBucketThreads));
#pragma unroll
        for (int u = 0; u < kU; u++) {
            atomicAdd(&lh[v[u].x >> shift], 1u);
            atomicAdd(&lh[v[u].y >> shift], 1u);
            atomicAdd(&lh[v[u].z >> shift], 1u);
            atomicAdd(&lh[v[u].w >> shift], 1u);
        }
    }
    for (; i0v < m; i0v += 4u * kBucketThreads)
        for (uint32_t j = i0v; j < m && j < i0v + 4; j++) atomicAdd(&lh[k[j] >> shift], 1u);
    __syncthreads();
    uint32_t* o = tile_cnt + ((uint64_t)r * tiles + tile) * stride;
    for (int b = threadIdx.x; b < nb; b += kBucketThreads) o[b] = lh[b];
}

// One workgroup per rank: tile_cnt[r][t][b] becomes the keys of bucket b in r's tiles before t;
// prefix[r][b] = r's keys in buckets before b, b = 0 .. nb.  A rank's only tile has no keys
// before it: its counts lie in `prefix` itself (tile_cnt == prefix) and become the prefix in place.
static __global__ __launch_bounds__(kBucketThreads) void bucket_rank_scan_kernel(int nb, uint32_t tiles,
                                                                        uint32_t* tile_cnt, uint32_t* prefix) {
    __shared__ uint32_t part[kBucketThreads / kWave];
    const int r = blockIdx.x;
    uint32_t* pre = prefix + (uint64_t)r * (nb + 1);
    const bool only = tiles == 1;
    uint32_t* row = only ? pre : tile_cnt + (uint64_t)r * tiles * nb;
    uint32_t carry = 0;
    constexpr int kU = 8;
    for (int b0 = 0; b0 < nb; b0 += kBucketThreads) {
        const int b = b0 + threadIdx.x;
        uint32_t sum = 0;
        if (only) {
            if (b < nb) sum = row[b];
        } else if (b < nb) {
            for (uint32_t t0 = 0; t0 < tiles; t0 += kU) {
                uint32_t c[kU];
#pragma unroll
                for (int u = 0; u < kU; u++) c[u] = row[(uint64_t)(t0 + u < tiles ? t0 + u : t0) * nb + b];
#pragma unroll
                for (int u = 0; u < kU; u++) {
                    if (t0 + u >= tiles) break;
                    row[(uint64_t)(t0 + u) * nb + b] = sum;
                    sum += c[u];
                }
            }
        }
        uint32_t all;
        const uint32_t ex = block_excl_sum<kBucketThreads>(sum, part, &all);
        if (b < nb) pre[b] = carry + ex;
        carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) pre[nb] = carry;
}

// acc[b] = keys of all ranks in buckets 0 .. b.  One workgroup per 64 buckets: its waves sum
// P / 16 rows each.
static __global__ __launch_bounds__(kBucketThreads) void bucket_colsum_kernel(const uint32_t* prefix, int P, int nb,
                                                                     int64_t* acc) {
    constexpr int kWaves = kBucketThreads / kWave;
    __shared__ int64_t part[kWaves][kWave];
    const int l = lane(), w = threadIdx.x >> 6;
    const int b = blockIdx.x * kWave + l;
    const uint32_t* col = prefix + 1 + (b < nb ? b : nb - 1);
    int64_t s = 0;
#pragma unroll 32
    for (int r = w; r < P; r += kWaves) s += col[(uint64_t)r * (nb + 1)];
    part[w][l] = s;
    __syncthreads();
    if (w == 0 && b < nb) {
        for (int k = 1; k < kWaves; k++) s += part[k][l];
        acc[b] = s;
    }
}

// NPB splitters (is.c:721-751): rank j takes buckets until the running total reaches (j+1)*n,
// at least one bucket.  With f_j the first bucket whose running total reaches (j+1)*n, rank j's
// last bucket is i_j = max(f_j, i_{j-1} + 1) = j + max over k <= j of (f_k - k): a search and a
// prefix maximum instead of a walk over the buckets by one thread (130 us at 1024 buckets and
// 512 ranks, 56 us at 512 and 4).  One workgroup.  With acc == nullptr it sums the ranks'
// prefixes itself.
constexpr int kBucketMax = 4096;
static __global__ __launch_bounds__(kBucketThreads) void bucket_splitters_kernel(const int64_t* acc,
                                                                        const uint32_t* prefix, int P, int nb,
                                                                        int64_t n, int32_t* lo, int32_t* hi) {
    constexpr int kWaves = kBucketThreads / kWave;
    __shared__ int64_t s_acc[kBucketMax];
    __shared__ int32_t s_max[kWaves];
    const int t = threadIdx.x, l = lane(), w = t >> 6;
    for (int b = t; b < nb; b += kBucketThreads) {
        int64_t s = 0;
        if (acc) {
            s = acc[b];
        } else {
#pragma unroll 8
            for (int r = 0; r < P; r++) s += prefix[(uint64_t)r * (nb + 1) + b + 1];
        }
        s_acc[b] = s;
    }
    __syncthreads();
    int32_t carry = INT32_MIN;       // max of f_k - k over the ranks of the passes before
    for (int j0 = 0; j0 < P; j0 += kBucketThreads) {
        const int j = j0 + t;
        int32_t v = INT32_MIN;
        if (j < P) {
            const int64_t want = (int64_t)(j + 1) * n;
            int a = 0, e = nb;       // first bucket with s_acc >= want, nb if none
            while (a < e) {
                const int mid = (a + e) >> 1;
                if (s_acc[mid] >= want) e = mid; else a = mid + 1;
            }
            v = a - j;
        }
        int32_t inc = v;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int32_t u = __shfl_up(inc, o);
            if (l >= o && u > inc) inc = u;
        }
        if (l == kWave - 1) s_max[w] = inc;
        __syncthreads();
        int32_t before = carry;
        for (int k = 0; k < kWaves; k++) {
            const int32_t x = s_max[k];
            if (k < w && x > before) before = x;
            if (x > carry) carry = x;
        }
        const int32_t up = __shfl_up(inc, 1);
        const int32_t prev = l > 0 && up > before ? up : before;    // over the ranks before j
        const int32_t upto = v > prev ? v : prev;
        if (j < P) {
            const int64_t last = (int64_t)j + upto;
            const bool some = last < nb;
            lo[j] = !some ? 1 : j == 0 ? 0 : (int32_t)((int64_t)j - 1 + prev + 1);
            hi[j] = some ? (int32_t)last : 0;
        }
        __syncthreads();
    }
}

__device__ __forceinline__ uint32_t bucket_of(uint32_t key, int shift, uint32_t buckets) {
    const uint32_t b = key >> shift;
    return b < buckets ? b : buckets - 1;
}

// The lanes whose b has the same low BITS bits as this lane's.  Four VALU
// instructions per bit: the bit as a lane mask, its ballot, and same & ~(ballot ^ bit) on each
// half.  (From C the compiler makes eight: it compares and selects instead of keeping the mask.)
template <int BITS>
__device__ __forceinline__ uint64_t same_bucket(uint32_t b) {
    uint32_t lo = ~0u, hi = ~0u;
#pragma unroll
    for (int q = 0; q < BITS; q++) {
        int32_t bit;
        asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(bit) : "v"(b), "n"(q));
        const uint64_t on = ballot(bit != 0);
        lo = __builtin_amdgcn_bitop3_b32(lo, (uint32_t)on, (uint32_t)bit, 0x90);
        hi = __builtin_amdgcn_bitop3_b32(hi, (uint32_t)(on >> 32), (uint32_t)bit, 0x90);
    }
    return (uint64_t)hi << 32 | lo;
}

__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Stable bucketing (is.c:680-688) of one tile of NT * KPT keys.  Wave w holds the tile's keys
// [w * 64 * KPT, +64 * KPT), 64 consecutive ones per register.  A key's place among the tile's
// keys of its bucket is: those of the waves before (a column of `cnt`), those of the wave's
// registers before (the running count in `cnt`), and those of the lanes before (the lanes with
// the same bucket, from one ballot per bucket bit).  The keys are then put in order in LDS and
// leave it in runs of one bucket, so that a wave's store covers a few lines instead of 64.
// NBC: buckets provided for (1024 or 4096, whose per-wave counters need the LDS of half as many
// waves).  The ballots (4 VALU instructions per bit) and HBM bound it about alike.
// TURNS: the workgroup takes `subs` tiles in turn and moves its row of tile_off (of prefix, if the
// rank has no other workgroup) on after each; apart, since the loop costs the single tile 1.5 %.
template <int NT, int KPT, int NBC, bool TURNS>
static __global__ __launch_bounds__(NT, NT == 1024 ? 8 : 4) void bucket_scatter_kernel(const uint32_t* keys, int P, int64_t n, int shift,
                                                            int nb, uint32_t tiles, uint32_t subs, uint32_t* tile_off,
                                                            uint32_t* prefix, const int32_t* lo,
                                                            const int32_t* hi, uint32_t* out, int32_t* scounts,
                                                            int32_t* sdispls) {
    constexpr int kWaves = NT / kWave, kTile = NT * KPT, kPer = NBC / NT;
    constexpr int kBits = NBC == 1024 ? 10 : 12;
    static_assert(NBC == (1 << kBits) && kTile <= 65536 && kPer >= 1 && KPT % 2 == 0, "tile positions fit 16 bits");
    constexpr size_t kCnt = sizeof(uint16_t) * kWaves * NBC, kOrd = sizeof(uint32_t) * kTile;
    __shared__ alignas(16) unsigned char pool[kCnt > kOrd ? kCnt : kOrd];   // counters, then the ordered keys
    __shared__ uint32_t gbase[NBC];       // global index of tile position 0, per bucket
    __shared__ uint32_t part[kWaves];
    uint16_t(*cnt)[NBC] = (uint16_t(*)[NBC])pool;
    uint32_t* ordered = (uint32_t*)pool;
    int r;
    uint32_t tile;
    if (!bucket_tile_of(blockIdx.x, P, tiles, &r, &tile)) return;
    uint32_t* pre = prefix + (uint64_t)r * (nb + 1);
    uint32_t* off = tiles > 1 ? tile_off + ((uint64_t)r * tiles + tile) * nb : nullptr;
    if (tile == 0) {
        for (int d = threadIdx.x; d < P; d += NT) {
            const int a = lo[d], b = hi[d];
            const bool some = a <= b;
            scounts[(int64_t)r * P + d] = some ? (int32_t)(pre[b + 1] - pre[a]) : 0;
            sdispls[(int64_t)r * P + d] = some ? (int32_t)pre[a] : (int32_t)pre[nb];
        }
    }
    uint32_t* o = out + (int64_t)r * n;
    for (uint32_t sub = 0;; sub++) {
        int t = threadIdx.x;
        if constexpr (TURNS) asm volatile("" : "+v"(t));   // addresses anew for each tile: kept over the loop, they would spill
        const int l = t & (kWave - 1), w = t >> 6;
        const int64_t i0 = (TURNS ? (int64_t)tile * subs + sub : (int64_t)tile) * kTile;
        const uint32_t m = (uint32_t)(n - i0 < kTile ? n - i0 : kTile);
        const uint32_t* k = keys + (int64_t)r * n + i0;
        const uint32_t first = (uint32_t)(w * kWave * KPT + l);
        uint32_t key[KPT], pos[KPT / 2] = {};   // positions: 16 bits each
#pragma unroll
        for (int i = 0; i < KPT; i++) {
            const uint32_t j = first + i * kWave;
            const uint32_t v = k[j < m ? j : 0];
            // past the last key: the last bucket's last places, which are never stored
            key[i] = j < m ? v : 0xFFFFFFFFu;
        }
        for (uint32_t z = t; z < kCnt / 4; z += NT) ((uint32_t*)pool)[z] = 0;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < KPT; i++) {
            const uint32_t b = bucket_of(key[i], shift, NBC);
            const uint64_t same = same_bucket<kBits>(b);
            const uint32_t at = cnt[w][b];
            __builtin_amdgcn_wave_barrier();
            // every lane of a group of equal buckets stores the same count
            cnt[w][b] = (uint16_t)(at + (uint32_t)__popcll(same));
            __builtin_amdgcn_wave_barrier();
            pos[i / 2] |= (at + lanes_below(same)) << (16 * (i & 1));
            asm volatile("" : "+v"(pos[i / 2]));   // now: the masks of 16 keys kept for later would spill
        }
        __syncthreads();
        // thread t: buckets t * kPer .. +kPer; their counts per wave become positions in the tile
        uint32_t tot[kPer], sum = 0;
#pragma unroll
        for (int q = 0; q < kPer; q++) {
            const int b = t * kPer + q;
            uint32_t run = 0;
#pragma unroll
            for (int u = 0; u < kWaves; u++) {
                const uint32_t c = cnt[u][b];
                cnt[u][b] = (uint16_t)run;
                run += c;
            }
            tot[q] = run;
            sum += run;
        }
        uint32_t all;
        uint32_t start = block_excl_sum<NT>(sum, part, &all);
        const bool more = TURNS && sub + 1 < subs && i0 + kTile < n;
#pragma unroll
        for (int q = 0; q < kPer; q++) {
            const int b = t * kPer + q;
#pragma unroll
            for (int u = 0; u < kWaves; u++) cnt[u][b] = (uint16_t)(cnt[u][b] + start);
            const uint32_t p0 = b < nb ? pre[b] : 0u, p1 = off && b < nb ? off[b] : 0u;
            gbase[b] = p0 + p1 - start;
            if (more && b < nb) {       // the next tile's keys of the bucket follow (only this workgroup reads the word)
                if (off) off[b] = p1 + tot[q];
                else pre[b] = p0 + tot[q];
            }
            start += tot[q];
        }
        __syncthreads();
        asm volatile("" : "+s"(shift));   // recompute the buckets: kept, they would spill at 64 registers
#pragma unroll
        for (int i = 0; i < KPT; i++) pos[i / 2] += (uint32_t)cnt[w][bucket_of(key[i], shift, NBC)] << (16 * (i & 1));
        __syncthreads();   // the counters' LDS takes the ordered keys
#pragma unroll
        for (int i = 0; i < KPT; i++)
            ordered[pos[i / 2] >> (16 * (i & 1)) & 0xFFFFu] = key[i];
        __syncthreads();
        if (m == kTile) {
#pragma unroll
            for (int i = 0; i < KPT; i++) {
                const uint32_t p = (uint32_t)(t + i * NT);
                const uint32_t v = ordered[p];
                o[gbase[v >> shift] + p] = v;
            }
        } else {
#pragma unroll
            for (int i = 0; i < KPT; i++) {
                const uint32_t p = (uint32_t)(t + i * NT);
                if (p < m) {
                    const uint32_t v = ordered[p];
                    o[gbase[v >> shift] + p] = v;
                }
            }
        }
        if (!more) return;
        __syncthreads();     // the next tile's counters take the LDS
    }
}

// ------------------------------------------------------------------ local sort
// Every rank owns a disjoint, ascending key range (the bucket ranges), so the local
// sorts of all ranks together are one counting sort of the concatenated receive buffers:
// rank d's sorted keys are the slice [recv_off_d, recv_off_d + recv_tot_d) of the output.
//
// Keys of at most kSortLowBits bits: workgroups count their keys in LDS and add the counts to
// one table (sort_count), then every workgroup scans the table and writes a range of the
// output (sort_expand).  Keys of up to kSortLowBits + kSortTopBits bits are first split by
// their top bits into parts of 2^kSortLowBits values: sort_top_hist and sort_top_scan place
// the parts, sort_split moves each key's low 16 bits into its part -- the part's own
// place in the output, whose 4 bytes per key hold 2, so no buffer of the keys' size is needed --
// and sort_part counts and rewrites each part in place, one workgroup per part.  Parts with
// more keys than one workgroup should take (skewed keys) are counted by several workgroups
// into a table and written by sort_part_expand.  HBM traffic 16 B per key (4 read twice, 2
// written, 2 read, 4 written).  Measured for 2^27 uniform keys below 2^23 as the bucket
// exchange leaves them: top_hist 94 us, split 254, part 170.  Counting with an atomic per key
// on 2^23 counters in HBM, and writing each value's run with one thread, took 4731 + 580 us.
// Longer keys, and an output that overlaps the keys (the split would overwrite keys not
// yet read), keep the counters in HBM (sort_hist and what follows it).
constexpr int kSortLowBits = 14;
constexpr int kSortTopBits = 10;
constexpr int kSortBins = 1 << kSortLowBits;
constexpr int kSortParts = 1 << kSortTopBits;
constexpr int kSortThreads = 1024;
constexpr int kSortTile = 16 * kSortThreads;   // keys per workgroup of the split; outputs per pass of the expansion

typedef u32x4 sort_u32x4_a2 __attribute__((aligned(2)));

// The split sort's tables (device memory): keys per part, first output of the part, keys moved
// so far; work items before the part; table number of the part (-1: one workgroup counts it).
struct SortParts {
    uint32_t* count;     // [parts]
    uint32_t* first;     // [parts + 1]
    uint32_t* moved;     // [parts]
    uint32_t* item;      // [parts + 1]
    int32_t* table;      // [parts]
    uint32_t* tables;    // [ntables][kSortBins]
};

// Work items of a part of c keys, and the end of its item that starts at key i0 < c.  A part
// may hold nearly 2^32 keys: a sum with `chunk` before the division or comparison would wrap,
// and the part's last item, or the whole part, would be left out.
__host__ __device__ __forceinline__ uint32_t sort_items(uint32_t c, uint32_t most, uint32_t chunk) {
    return c > most ? (c - 1) / chunk + 1 : c ? 1 : 0;
}
__host__ __device__ __forceinline__ uint32_t sort_item_end(uint32_t i0, uint32_t c, uint32_t chunk) {
    return c - i0 < chunk ? c : i0 + chunk;
}

static __global__ __launch_bounds__(kSortThreads) void sort_zero_kernel(uint32_t* p, uint32_t words) {
    for (uint32_t i = blockIdx.x * kSortThreads + threadIdx.x; i < words; i += gridDim.x * kSortThreads) p[i] = 0;
}

// Adds 1 to lds[b] for every valid lane and returns the lane's place among them.  The lanes that
// share the first valid lane's b add once, then those that share the next one's (the keys of one
// rank's slice fall into one or two parts, and LDS adds to one word go one by one), the rest
// each for itself.
__device__ __forceinline__ uint32_t lds_count(uint32_t* lds, uint32_t b, bool valid) {
    uint32_t place = 0;
    uint64_t left = ballot(valid);
#pragma unroll
    for (int round = 0; round < 2; round++) {
        if (!left) return place;      // wave-uniform
        const int lead = __builtin_ctzll(left);
        const bool mine = (left >> lane() & 1) && b == readlane(b, lead);
        const uint64_t same = ballot(mine);
        uint32_t at = 0;
        if (lane() == lead) at = atomicAdd(&lds[b], (uint32_t)__popcll(same));
        at = readlane(at, lead) + lanes_below(same);
        if (mine) place = at;
        left &= ~same;
    }
    if (left >> lane() & 1) place = atomicAdd(&lds[b], 1u);
    return place;
}

// Whether the wave's N keys per lane (those below the lane's `live`) lie in at most two parts, a
// and b (b = a if in one); every lane's first key must be live.
template <int N>
__device__ __forceinline__ bool sort_two_parts(const uint32_t (&part)[N], const bool (&live)[N], uint32_t* a, uint32_t* b) {
    const uint32_t a0 = bcast(part[0]);
    uint32_t other = a0;
#pragma unroll
    for (int i = 0; i < N; i++) other = live[i] && part[i] != a0 ? part[i] : other;
    const uint64_t have = ballot(other != a0);
    const uint32_t b0 = have ? readlane(other, __builtin_ctzll(have)) : a0;
    bool ok = true;
#pragma unroll
    for (int i = 0; i < N; i++) ok = ok && (!live[i] || part[i] == a0 || part[i] == b0);
    *a = a0;
    *b = b0;
    return ballot(!ok) == 0;
}

// Four keys per lane counted by their parts; one add per part where the wave has one or two.
__device__ __forceinline__ void sort_count_parts(uint32_t* lds, u32x4 v) {
    const uint32_t b[4] = {v.x >> kSortLowBits, v.y >> kSortLowBits, v.z >> kSortLowBits, v.w >> kSortLowBits};
    const bool live[4] = {true, true, true, true};
    uint32_t p, q;
    if (sort_two_parts(b, live, &p, &q)) {
        const uint64_t act = ballot(true);
        uint32_t np = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) np += (uint32_t)__popcll(ballot(b[k] == p));
        const uint32_t nq = 4u * (uint32_t)__popcll(act) - np;
        if (lane() == (int)__builtin_ctzll(act)) {
            atomicAdd(&lds[p], np);
            if (nq) atomicAdd(&lds[q], nq);
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) lds_count(lds, b[k], true);
    }
}

// keys >> kSortLowBits counted into part counts; workgroup g takes keys [g * per, +per), per a
// multiple of 4 * kSortThreads.
static __global__ __launch_bounds__(kSortThreads) void sort_top_hist_kernel(const uint32_t* keys, int64_t n, int64_t per,
                                                                   uint32_t parts, uint32_t* count) {
    __shared__ uint32_t lh[kSortParts];
    for (uint32_t b = threadIdx.x; b < parts; b += kSortThreads) lh[b] = 0;
    __syncthreads();
    const int64_t i0 = (int64_t)blockIdx.x * per, i1 = i0 + per < n ? i0 + per : n;
    int64_t i = i0 + 4 * (int64_t)threadIdx.x;
    constexpr int kU = 4;       // 16-byte loads in flight per thread
    for (; i0 + per <= n && i + 4 * (kU - 1) * kSortThreads < i1; i += 4 * kU * kSortThreads) {
        u32x4 v[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) v[u] = gload16((uint64_t)(uintptr_t)(keys + i + 4 * u * kSortThreads));
#pragma unroll
        for (int u = 0; u < kU; u++) sort_count_parts(lh, v[u]);
    }
    for (; i + 4 <= i1; i += 4 * kSortThreads) sort_count_parts(lh, gload16((uint64_t)(uintptr_t)(keys + i)));
    for (int64_t j = i; j < i1 && j < i + 4; j++) atomicAdd(&lh[keys[j] >> kSortLowBits], 1u);
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < parts; b += kSortThreads)
        if (lh[b]) atomicAdd(&count[b], lh[b]);
}

// One workgroup: where each part starts, its work items, and its table if it needs one.
static __global__ __launch_bounds__(kSortThreads) void sort_top_scan_kernel(SortParts s, uint32_t parts, uint32_t most,
                                                                   uint32_t chunk) {
    static_assert(kSortParts == kSortThreads, "one thread per part");
    __shared__ uint32_t part[kSortThreads / kWave];
    const uint32_t b = threadIdx.x;
    const uint32_t c = b < parts ? s.count[b] : 0;
    const bool big = c > most;
    const uint32_t items = sort_items(c, most, chunk);
    uint32_t all, nitem, nbig;
    const uint32_t first = block_excl_sum<kSortThreads>(c, part, &all);
    __syncthreads();
    const uint32_t item = block_excl_sum<kSortThreads>(items, part, &nitem);
    __syncthreads();
    const uint32_t slot = block_excl_sum<kSortThreads>(big ? 1u : 0u, part, &nbig);
    if (b < parts) {
        s.first[b] = first;
        s.item[b] = item;
        s.moved[b] = 0;
        s.table[b] = big ? (int32_t)slot : -1;
        if (b == parts - 1) {
            s.first[parts] = all;
            s.item[parts] = nitem;
        }
    }
}

// The low 16 bits of one tile's keys to their parts.  Part b's keys are 2-byte words at the
// start of out[first[b] .. first[b + 1]).  The order within a part does not matter.
static __global__ __launch_bounds__(kSortThreads, 8) void sort_split_kernel(const uint32_t* keys, int64_t n, SortParts s,
                                                                uint32_t parts, uint32_t ntables, uint32_t* out) {
    constexpr int kPer = kSortTile / kSortThreads;   // keys per thread, 4 consecutive ones per load
    __shared__ uint32_t cnt[kSortParts];
    __shared__ uint32_t at[kSortParts];       // place in the part of tile position 0
    __shared__ uint32_t base[kSortParts];     // first output of the part
    __shared__ uint32_t part[kSortThreads / kWave];
    __shared__ uint32_t ordered[kSortTile];
    const int t = threadIdx.x;
    // the tables of large parts start at zero (they are counted by the next kernel)
    for (uint64_t z = (uint64_t)blockIdx.x * kSortThreads + t; z < (uint64_t)ntables * kSortBins;
         z += (uint64_t)gridDim.x * kSortThreads)
        s.tables[z] = 0;
    const int64_t i0 = (int64_t)blockIdx.x * kSortTile;
    const uint32_t m = (uint32_t)(n - i0 < kSortTile ? n - i0 : kSortTile);
    uint32_t key[kPer];
    // key 4 q + j of a thread: tile index 4 (q * threads + t) + j
#pragma unroll
    for (int q = 0; q < kPer / 4; q++) {
        const uint32_t j = 4u * (uint32_t)(q * kSortThreads + t);
        if (j + 4 <= m) {
            const u32x4 v = gload16((uint64_t)(uintptr_t)(keys + i0 + j));
            key[4 * q] = v.x; key[4 * q + 1] = v.y; key[4 * q + 2] = v.z; key[4 * q + 3] = v.w;
        } else {
#pragma unroll
            for (int x = 0; x < 4; x++) key[4 * q + x] = keys[i0 + (j + x < m ? j + x : 0)];
        }
    }
    const uint32_t b0 = keys[i0] >> kSortLowBits;
    bool one = true;
#pragma unroll
    for (int i = 0; i < kPer; i++) one = one && (key[i] >> kSortLowBits) == b0;
    if (__syncthreads_and(one)) {
        // the whole tile in one part (the usual tile of concatenated receive buffers)
        if (t == 0) part[0] = atomicAdd(&s.moved[b0], m);
        __syncthreads();
        uint16_t* o = (uint16_t*)(out + s.first[b0]) + part[0];
#pragma unroll
        for (int q = 0; q < kPer / 4; q++) {
            const uint32_t j = 4u * (uint32_t)(q * kSortThreads + t);
            if (j + 4 <= m) {
                typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
                *(u32x2_a2*)(o + j) = u32x2_a2{(key[4 * q] & 0xFFFFu) | key[4 * q + 1] << 16,
                                               (key[4 * q + 2] & 0xFFFFu) | key[4 * q + 3] << 16};
            } else {
                for (int x = 0; x < 4; x++)
                    if (j + x < m) o[j + x] = (uint16_t)key[4 * q + x];
            }
        }
        return;
    }
    cnt[t] = 0;
    __syncthreads();
    uint32_t rank[kPer];
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const uint32_t j = 4u * (uint32_t)((i >> 2) * kSortThreads + t) + (i & 3);
        rank[i] = lds_count(cnt, key[i] >> kSortLowBits, j < m);
    }
    __syncthreads();
    const uint32_t c = cnt[t];
    uint32_t all;
    const uint32_t start = block_excl_sum<kSortThreads>(c, part, &all);
    if ((uint32_t)t < parts) {
        at[t] = (c ? atomicAdd(&s.moved[t], c) : 0u) - start;
        base[t] = s.first[t];
    }
    cnt[t] = start;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const uint32_t j = 4u * (uint32_t)((i >> 2) * kSortThreads + t) + (i & 3);
        if (j < m) ordered[cnt[key[i] >> kSortLowBits] + rank[i]] = key[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const uint32_t p = (uint32_t)(t + i * kSortThreads);
        if (p < m) {
            const uint32_t v = ordered[p], b = v >> kSortLowBits;
            ((uint16_t*)(out + base[b]))[at[b] + p] = (uint16_t)v;
        }
    }
}

// Writes outputs [q0, q1) of the sorted keys of a part of kSortBins values: value base + v
// count[v] times.  `count` may lie in LDS over `marks` (it is read first).  Thread t owns values
// 16 t .. 16 t + 15.  The output is written in tiles that start at 128-byte lines: each value
// marks the tile position where its run starts (or the tile's first position if it runs into
// the tile), a running maximum over the tile turns the marks into values, and the tile leaves
// LDS as coalesced 16-byte stores.  All kSortThreads threads call.
__device__ __forceinline__ void sort_write_runs(const uint32_t* count, uint32_t bins, uint32_t base, uint32_t* out,
                                                uint32_t q0, uint32_t q1, uint16_t* marks, uint32_t* part) {
    constexpr int kPer = kSortBins / kSortThreads;
    constexpr int kWaves = kSortThreads / kWave;
    const int t = threadIdx.x, l = lane(), w = t >> 6;
    uint32_t c[kPer], sum = 0;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const uint32_t v = (uint32_t)(t * kPer + k);
        c[k] = v < bins ? count[v] : 0u;
        sum += c[k];
    }
    uint32_t all;
    const uint32_t s0 = block_excl_sum<kSortThreads>(sum, part, &all);
    const uint32_t s1 = s0 + sum;
    // tile i covers [i * kSortTile - lead, +kSortTile) + q0
    const uint32_t lead = (uint32_t)(((uintptr_t)(out + q0) >> 2) & 31u);
    const uint32_t span = q1 - q0 + lead;
    for (uint32_t p0 = 0; p0 < span; p0 += kSortTile) {
        const uint32_t lo = p0 ? q0 + p0 - lead : q0;              // outputs [lo, hi) are in the tile
        const uint32_t hi = span - p0 < kSortTile ? q1 : q0 + p0 + kSortTile - lead;
        const uint32_t skip = p0 ? 0u : lead;                      // tile position of output lo
        __syncthreads();
        ((u32x4*)marks)[2 * t] = u32x4{0u, 0u, 0u, 0u};
        ((u32x4*)marks)[2 * t + 1] = u32x4{0u, 0u, 0u, 0u};
        __syncthreads();
        if (s0 < hi && s1 > lo) {
            uint32_t s = s0;
#pragma unroll
            for (int k = 0; k < kPer; k++) {
                const uint32_t e = s + c[k];
                if (c[k] && s < hi && e > lo) marks[skip + (s > lo ? s - lo : 0u)] = (uint16_t)(t * kPer + k + 1);
                s = e;
            }
        }
        __syncthreads();
        uint32_t word[8];
        {
            const u32x4 a = ((const u32x4*)marks)[2 * t], b = ((const u32x4*)marks)[2 * t + 1];
            word[0] = a.x; word[1] = a.y; word[2] = a.z; word[3] = a.w;
            word[4] = b.x; word[5] = b.y; word[6] = b.z; word[7] = b.w;
        }
        uint32_t run = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t x = word[k] & 0xFFFFu, y = word[k] >> 16;
            run = x > run ? x : run;
            const uint32_t a = run;
            run = y > run ? y : run;
            word[k] = a | run << 16;
        }
        uint32_t inc = run;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const uint32_t u = (uint32_t)__shfl_up((int)inc, o);
            if (l >= o && u > inc) inc = u;
        }
        if (l == kWave - 1) part[w] = inc;
        const uint32_t up = (uint32_t)__shfl_up((int)inc, 1);
        __syncthreads();
        uint32_t carry = l > 0 ? up : 0u;
#pragma unroll
        for (int k = 0; k < kWaves; k++) {
            const uint32_t x = part[k];
            if (k < w && x > carry) carry = x;
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
            uint32_t x = word[k] & 0xFFFFu, y = word[k] >> 16;
            x = x > carry ? x : carry;
            y = y > carry ? y : carry;
            word[k] = x | y << 16;
        }
        ((u32x4*)marks)[2 * t] = u32x4{word[0], word[1], word[2], word[3]};
        ((u32x4*)marks)[2 * t + 1] = u32x4{word[4], word[5], word[6], word[7]};
        __syncthreads();
        const uint32_t end = hi - lo + skip;                       // tile positions [skip, end)
        uint32_t* o = out + lo - skip;                             // tile position 0
        const uint32_t add = base - 1u;                            // marks hold value + 1
#pragma unroll
        for (int j = 0; j < kSortTile / (4 * kSortThreads); j++) {
            const uint32_t p = 4u * (uint32_t)(j * kSortThreads + t);
            if (p >= end) continue;
            const uint32_t x = ((const uint32_t*)marks)[p / 2], y = ((const uint32_t*)marks)[p / 2 + 1];
            const u32x4 v{(x & 0xFFFFu) + add, (x >> 16) + add, (y & 0xFFFFu) + add, (y >> 16) + add};
            if (p >= skip && p + 4 <= end) {
                *(u32x4*)(o + p) = v;
            } else {
                const uint32_t e[4] = {v.x, v.y, v.z, v.w};
                for (int k = 0; k < 4; k++)
                    if (p + k >= skip && p + k < end) o[p + k] = e[k];
            }
        }
    }
}

// The part that holds work item g, and which of its items g is.
__device__ __forceinline__ uint32_t sort_part_of(const SortParts& s, uint32_t parts, uint32_t g, uint32_t* nth) {
    uint32_t a = 0, e = parts;      // last part with item[b] <= g; empty parts share it with the next
    while (e - a > 1) {
        const uint32_t mid = (a + e) >> 1;
        if (s.item[mid] <= g) a = mid; else e = mid;
    }
    *nth = g - s.item[a];
    return a;
}

// One workgroup per work item: a whole part is counted in LDS and rewritten as its sorted
// values; a piece of a large part is counted and added to the part's table.
static __global__ __launch_bounds__(kSortThreads, 8) void sort_part_kernel(SortParts s, uint32_t parts, uint32_t chunk,
                                                               uint32_t* out) {
    __shared__ alignas(16) uint32_t hist[kSortBins];
    __shared__ uint32_t part[kSortThreads / kWave];
    if (blockIdx.x >= s.item[parts]) return;
    uint32_t nth;
    const uint32_t b = sort_part_of(s, parts, blockIdx.x, &nth);
    const uint32_t first = s.first[b], c = s.first[b + 1] - first;
    const int32_t table = s.table[b];
    const uint32_t i0 = table < 0 ? 0 : nth * chunk;
    const uint32_t m = (table < 0 ? c : sort_item_end(i0, c, chunk)) - i0;
    const int t = threadIdx.x;
    for (int k = t; k < kSortBins; k += kSortThreads) hist[k] = 0;
    __syncthreads();
    const uint16_t* k16 = (const uint16_t*)(out + first) + i0;
    constexpr uint32_t kLow = kSortBins - 1;
    uint32_t i = 8u * (uint32_t)t;
    for (; i + 8 <= m; i += 8 * kSortThreads) {
        const u32x4 v = *(const sort_u32x4_a2*)(k16 + i);
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            atomicAdd(&hist[x[k] & kLow], 1u);
            atomicAdd(&hist[(x[k] >> 16) & kLow], 1u);
        }
    }
    for (uint32_t j = i; j < m && j < i + 8; j++) atomicAdd(&hist[k16[j] & kLow], 1u);
    __syncthreads();
    if (table < 0) {
        sort_write_runs(hist, kSortBins, b << kSortLowBits, out + first, 0, c, (uint16_t*)hist, part);
        return;
    }
    uint32_t* to = s.tables + (uint64_t)table * kSortBins;
    for (int k = t; k < kSortBins; k += kSortThreads)
        if (hist[k]) atomicAdd(&to[k], hist[k]);
}

// The outputs of the large parts, one work item's range per workgroup.
static __global__ __launch_bounds__(kSortThreads, 8) void sort_part_expand_kernel(SortParts s, uint32_t parts, uint32_t chunk,
                                                                      uint32_t* out) {
    __shared__ alignas(16) uint16_t marks[kSortTile];
    __shared__ uint32_t part[kSortThreads / kWave];
    if (blockIdx.x >= s.item[parts]) return;
    uint32_t nth;
    const uint32_t b = sort_part_of(s, parts, blockIdx.x, &nth);
    const int32_t table = s.table[b];
    if (table < 0) return;
    const uint32_t first = s.first[b], c = s.first[b + 1] - first;
    const uint32_t i0 = nth * chunk, i1 = sort_item_end(i0, c, chunk);
    sort_write_runs(s.tables + (uint64_t)table * kSortBins, kSortBins, b << kSortLowBits, out + first, i0, i1, marks,
                    part);
}

// Short keys: counts of keys [g * per, +per) added to hist[bins].
static __global__ __launch_bounds__(kSortThreads) void sort_count_kernel(const uint32_t* keys, int64_t n, int64_t per,
                                                                uint32_t bins, uint32_t* hist) {
    __shared__ uint32_t lh[kSortBins];
    for (uint32_t b = threadIdx.x; b < bins; b += kSortThreads) lh[b] = 0;
    __syncthreads();
    const int64_t i0 = (int64_t)blockIdx.x * per, i1 = i0 + per < n ? i0 + per : n;
    int64_t i = i0 + 4 * (int64_t)threadIdx.x;
    for (; i + 4 <= i1; i += 4 * kSortThreads) {
        const u32x4 v = gload16((uint64_t)(uintptr_t)(keys + i));
        atomicAdd(&lh[v.x], 1u);
        atomicAdd(&lh[v.y], 1u);
        atomicAdd(&lh[v.z], 1u);
        atomicAdd(&lh[v.w], 1u);
    }
    for (int64_t j = i; j < i1 && j < i + 4; j++) atomicAdd(&lh[keys[j]], 1u);
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < bins; b += kSortThreads)
        if (lh[b]) atomicAdd(&hist[b], lh[b]);
}

// Short keys: workgroup g writes outputs [g * per, +per).
static __global__ __launch_bounds__(kSortThreads, 8) void sort_expand_kernel(const uint32_t* hist, uint32_t bins, int64_t n,
                                                                 int64_t per, uint32_t* out) {
    __shared__ alignas(16) uint16_t marks[kSortTile];
    __shared__ uint32_t part[kSortThreads / kWave];
    const int64_t q0 = (int64_t)blockIdx.x * per, q1 = q0 + per < n ? q0 + per : n;
    sort_write_runs(hist, bins, 0, out, (uint32_t)q0, (uint32_t)q1, marks, part);
}

constexpr int kSortLdsBins = 16384;  // keys below this are counted in LDS first

static __global__ void __launch_bounds__(1024) sort_hist_kernel(const uint32_t* keys, int64_t n,
                                                         uint32_t nbins, uint32_t* hist) {
    __shared__ uint32_t lh[kSortLdsBins];
    const uint32_t lds_bins = nbins < kSortLdsBins ? nbins : kSortLdsBins;
    for (uint32_t b = threadIdx.x; b < lds_bins; b += blockDim.x) lh[b] = 0;
    __syncthreads();
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t k = keys[i];
        if (k < lds_bins) atomicAdd(&lh[k], 1u);
        else atomicAdd(&hist[k], 1u);
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < lds_bins; b += blockDim.x)
        if (lh[b]) atomicAdd(&hist[b], lh[b]);
}

// Exclusive scan of nbins counters in three kernels (4096 counters per 1024-thread block).
static __global__ void __launch_bounds__(1024) scan_block_sums_kernel(const uint32_t* h, uint32_t nbins,
                                                               uint64_t* sums) {
    __shared__ uint64_t red[16];
    const uint64_t base = (uint64_t)blockIdx.x * 4096;
    uint64_t s = 0;
    for (int k = 0; k < 4; k++) {
        const uint64_t i = base + (uint64_t)k * 1024 + threadIdx.x;
        if (i < nbins) s += h[i];
    }
    s = (uint64_t)wave_sum((int64_t)s);
    if (lane() == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t t = 0;
        for (int w = 0; w < 16; w++) t += red[w];
        sums[blockIdx.x] = t;
    }
}

static __global__ void __launch_bounds__(1024) scan_sums_kernel(uint64_t* sums, int nblocks) {
    // single block, exclusive scan in place (sequential chunks of 1024)
    __shared__ uint64_t part[16];
    uint64_t carry = 0;
    for (int base = 0; base < nblocks; base += 1024) {
        const int i = base + threadIdx.x;
        const uint64_t v = i < nblocks ? sums[i] : 0;
        const uint64_t inc = (uint64_t)wave_incl_scan((int64_t)v);
        if (lane() == 63) part[threadIdx.x >> 6] = inc;
        __syncthreads();
        uint64_t before = 0;
        for (int w = 0; w < (int)(threadIdx.x >> 6); w++) before += part[w];
        uint64_t total = 0;
        for (int w = 0; w < 16; w++) total += part[w];
        if (i < nblocks) sums[i] = carry + before + inc - v;
        carry += total;
        __syncthreads();
    }
}

static __global__ void __launch_bounds__(1024) scan_apply_kernel(const uint32_t* h, uint32_t nbins,
                                                          const uint64_t* sums, uint32_t* prefix) {
    __shared__ uint64_t part[16];
    const uint64_t base = (uint64_t)blockIdx.x * 4096;
    uint64_t carry = sums[blockIdx.x];
    for (int k = 0; k < 4; k++) {
        const uint64_t i = base + (uint64_t)k * 1024 + threadIdx.x;
        const uint64_t v = i < nbins ? h[i] : 0;
        const uint64_t inc = (uint64_t)wave_incl_scan((int64_t)v);
        if (lane() == 63) part[threadIdx.x >> 6] = inc;
        __syncthreads();
        uint64_t before = 0, total = 0;
        for (int w = 0; w < 16; w++) {
            if (w < (int)(threadIdx.x >> 6)) before += part[w];
            total += part[w];
        }
        if (i < nbins) prefix[i] = (uint32_t)(carry + before + inc - v);
        carry += total;
        __syncthreads();
    }
}

// Writes each value's run; runs longer than 256 go to a list filled by whole blocks.
static __global__ void sort_runs_kernel(const uint32_t* hist, const uint32_t* prefix, uint32_t nbins,
                                 uint32_t* out, uint32_t* big, uint32_t* nbig) {
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nbins;
         v += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t c = hist[v];
        if (c == 0) continue;
        if (c <= 256) {
            const uint32_t o = prefix[v];
            for (uint32_t k = 0; k < c; k++) out[o + k] = (uint32_t)v;
        } else {
            big[atomicAdd(nbig, 1u)] = (uint32_t)v;
        }
    }
}

static __global__ void sort_fill_runs_kernel(const uint32_t* hist, const uint32_t* prefix,
                                      const uint32_t* big, const uint32_t* nbig, uint32_t* out) {
    const uint32_t nb = *nbig;
    for (uint32_t r = blockIdx.x; r < nb; r += gridDim.x) {
        const uint32_t v = big[r];
        const uint32_t c = hist[v], o = prefix[v];
        for (uint32_t k = threadIdx.x; k < c; k += blockDim.x) out[o + k] = v;
    }
}

// Number of keys < bound in keys[0, n) (partial verification of NPB IS).
static __global__ void count_less_kernel(const uint32_t* keys, int64_t n, uint32_t bound,
                                  unsigned long long* out) {
    uint64_t c = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        c += keys[i] < bound;
    c = (uint64_t)wave_sum((int64_t)c);
    if (lane() == 0 && c) atomicAdd(out, (unsigned long long)c);
}

}  // namespace gpumpi
