// Batched point-to-point step: the matched Send/Recv pairs of one step as two kernels,
// replayable from a hipGraph.
//
// Semantics per pair: those of a matched MPI_Isend / MPI_Irecv pair (gpu_libc/
// cuda_mpi.cu:65-118, gpu_mpi/mpi.cu:617-645) once both have completed -- `bytes` bytes of
// the sender's buffer are in the receiver's.  The list is device memory and is read when
// the step runs, so a kernel earlier on the same stream (or in the same graph) may write
// this step's pairs, sizes included.  Destinations must not overlap each other or any
// source (as MPI's receive buffers must not); zero-byte pairs are allowed.
//
// The reference moves each pair with one thread's memcpy after an envelope handshake.
// Here the step needs no handshake: the pair list is the match.  Work is cut at 8 KiB
// boundaries of each destination address ("chunks"), so every chunk's interior is
// 16-byte aligned on the store side whatever the buffers' alignment:
//   p2p_scan_kernel  exclusive prefix sums of the pairs' chunk counts within tiles of pairs, a
//                    workgroup per tile, and the tiles' totals;
//   p2p_copy_kernel  finds the pair of a chunk by 64-ary searches of the offsets and walks
//                    forward; a chunk is 8 unaligned 16-byte loads per lane, all issued before
//                    its stores.
// Lists of up to kP2pFused pairs need no scan kernel: every copy workgroup scans the whole list
// into LDS.  Measured against a scan by one workgroup and cached loads and stores throughout, us
// per step on three sets of buffers in turn: 3072 pairs of 5 KiB 14.6 -> 11.4, 65536 pairs of 4 KiB
// 189 -> 141 (their scan, by events, 56 -> 8), 1000 pairs of 256 KiB 119 -> 116, 64 pairs of 16
// MiB 440 -> 415.
// HBM traffic = 2 x the bytes of the pairs (read once, written once) + 8 B per pair of
// offsets (or, without a scan kernel, 24 B per pair and workgroup from the L2s: 16 workgroups per
// CU up to kP2pShort pairs, one up to kP2pFused).
#pragma once

#include "common.h"
#include "copy.h"

namespace gpumpi {

struct P2pPair {
    const char* src;
    char* dst;
    uint64_t bytes;
};

constexpr int kP2pChunkShift = 13;                       // 8 KiB chunks of the destination
constexpr uint64_t kP2pChunk = 1ull << kP2pChunkShift;
constexpr int kP2pU = (int)(kP2pChunk / 16 / kWave);     // 16-byte vectors per lane and chunk
constexpr int kP2pScanThreads = 1024;
constexpr int kP2pFused = 4096;      // pairs that every workgroup scans for itself
constexpr int kP2pShort = 256;       // and that even small workgroups do
constexpr int kP2pPass = 4096;       // pairs per pass of a tile's scan
constexpr int kP2pTiles = 1024;      // tiles at most: their totals are scanned into LDS

// Branch-free, so that callers can issue the loads of many pairs before using any.
__device__ __forceinline__ uint64_t p2p_chunks(const char* dst, uint64_t bytes) {
    const uint64_t a = (uint64_t)(uintptr_t)dst;
    const uint64_t c = ((a + bytes - 1) >> kP2pChunkShift) - (a >> kP2pChunkShift) + 1;
    return bytes ? c : 0;
}

// Exclusive sum of one value per thread over a workgroup of NT threads, and the total; `part`
// holds one word per wavefront and is free after the caller's next barrier.
template <int NT>
__device__ __forceinline__ uint64_t p2p_block_scan(uint64_t v, uint64_t* part, uint64_t* total) {
    constexpr int kWaves = NT / kWave;
    const int l = lane(), w = threadIdx.x >> 6;
    uint64_t incl = v;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const uint64_t u = __shfl_up(incl, o);
        if (l >= o) incl += u;
    }
    if (l == kWave - 1) part[w] = incl;
    __syncthreads();
    uint64_t before = 0, all = 0;
#pragma unroll
    for (int u = 0; u < kWaves; u++) {
        const uint64_t x = part[u];
        before += u < w ? x : 0;
        all += x;
    }
    *total = all;
    return before + incl - v;
}

// Chunk counts of pairs [i0, i0 + PASS) below i1 to exclusive offsets in s (LDS), from
// `carry` on; returns the carry after them.  The pairs are read coalesced and without a branch
// (a clamped index and a masked size: under a bounds branch each load would be waited for).
template <int NT, int PASS>
__device__ __forceinline__ uint64_t p2p_scan_pass(const P2pPair* pairs, int64_t i0, int64_t i1, uint64_t carry,
                                                  uint64_t* s, uint64_t* part) {
    constexpr int kPer = PASS / NT;
    const int t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int64_t j = i0 + (int64_t)k * NT + t;
        const P2pPair p = pairs[j < i1 ? j : i1 - 1];
        s[k * NT + t] = p2p_chunks(p.dst, j < i1 ? p.bytes : 0);
    }
    __syncthreads();
    uint64_t c[kPer], sum = 0, all;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        c[k] = s[t * kPer + k];
        sum += c[k];
    }
    uint64_t run = carry + p2p_block_scan<NT>(sum, part, &all);
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        s[t * kPer + k] = run;
        run += c[k];
    }
    __syncthreads();
    return carry + all;
}

// chunk_off[i] = chunks of the pairs before i in i's tile of 1 << tile_shift pairs;
// tile_chunks[b] = chunks of tile b.
static __global__ __launch_bounds__(kP2pScanThreads) void p2p_scan_kernel(const P2pPair* pairs, int64_t n, int tile_shift,
                                                               uint64_t* chunk_off, uint64_t* tile_chunks) {
    __shared__ uint64_t s_c[kP2pPass];
    __shared__ uint64_t s_w[kP2pScanThreads / kWave];
    const int64_t t0 = (int64_t)blockIdx.x << tile_shift, t1 = t0 + (1ll << tile_shift) < n ? t0 + (1ll << tile_shift) : n;
    uint64_t carry = 0;
    for (int64_t i0 = t0; i0 < t1; i0 += kP2pPass) {
        carry = p2p_scan_pass<kP2pScanThreads, kP2pPass>(pairs, i0, t1, carry, s_c, s_w);
#pragma unroll
        for (int k = 0; k < kP2pPass / kP2pScanThreads; k++) {
            const int64_t j = i0 + (int64_t)k * kP2pScanThreads + threadIdx.x;
            if (j < t1) chunk_off[j] = s_c[k * kP2pScanThreads + threadIdx.x];
        }
        __syncthreads();   // s_c is rewritten by the next pass
    }
    if (threadIdx.x == 0) tile_chunks[blockIdx.x] = carry;
}

// What a step leaves in the caches, by its size: up to kP2pLoads bytes everything; then only what
// it wrote, for its reader (the loads are non-temporal, so that the sent bytes do not push the
// received ones out); from kP2pStores on nothing.  A pair of b bytes anywhere covers b / 8 KiB + 1
// chunks on average.  Measured on three sets of buffers in turn, us for the step alone / with an
// elementwise pass over the received bytes / with the same step back:
//   pairs, size      all cached        stores cached        nothing       loads cached only
//   3072, 15 MiB   11.3  18.4  23.1   13.2  20.3  25.8         -          10.9  18.8  26.9
//   64, 40 MiB     15.2  31.7  30.7   17.3  32.0  37.4         -          15.5  35.3  37.2
//   1000, 56 MiB   28.7  47.3  51.6   25.5  44.5  53.8         -          23.1  51.2  57.1
//   3072, 96 MiB   48.8  85.0  94.3   44.0  77.6  81.5         -          43.4  83.1  94.2
//   64, 256 MiB     107   199   213    108   192   186         -           102   208   205
//   64, 512 MiB     211   397   421    215   397   429         -           204   400   407
//   64, 768 MiB     319   598    -            -           313  593  626    314   604   629
enum P2pCaching : int { kP2pCached = 0, kP2pKeepStores = 1, kP2pKeepNothing = 2 };
constexpr uint64_t kP2pLoads = 48u << 20, kP2pStores = 512u << 20;
__host__ __device__ __forceinline__ P2pCaching p2p_caching(uint64_t chunks, int64_t pairs) {
    if (chunks < (kP2pLoads >> kP2pChunkShift) + (uint64_t)pairs) return kP2pCached;
    return chunks < (kP2pStores >> kP2pChunkShift) + (uint64_t)pairs ? kP2pKeepStores : kP2pKeepNothing;
}

// Copies dst bytes [lo, hi) from the matching source bytes (one chunk or less, so at most
// kP2pU vectors per lane).  All 64 lanes call with the same arguments.
template <int C>
__device__ __forceinline__ void p2p_copy_piece(char* dst, const char* src, uint64_t lo, uint64_t hi) {
    const int l = lane();
    const uint64_t d0 = (uint64_t)(uintptr_t)dst;
    const uint64_t a = (lo + 15) & ~(uint64_t)15, b = hi & ~(uint64_t)15;
    if (a >= b) {   // no whole aligned vector: bytes
        for (uint64_t x = lo + (uint64_t)l; x < hi; x += kWave)
            *(char*)(uintptr_t)x = src[x - d0];
        return;
    }
    if ((uint64_t)l < a - lo) *(char*)(uintptr_t)(lo + l) = src[lo + l - d0];
    if ((uint64_t)l < hi - b) *(char*)(uintptr_t)(b + l) = src[b + l - d0];
    const uint64_t nvec = (b - a) >> 4;
    const uint64_t sa = (uint64_t)(uintptr_t)src + (a - d0);
    auto load = [](uint64_t at) { return C == kP2pCached ? gload16(at) : gload16_nt(at); };
    constexpr bool kNt = C == kP2pKeepNothing;
    u32x4 v[kP2pU];
    if (nvec == (uint64_t)kWave * kP2pU) {
#pragma unroll
        for (int u = 0; u < kP2pU; u++) v[u] = load(sa + 16 * ((uint64_t)u * kWave + l));
#pragma unroll
        for (int u = 0; u < kP2pU; u++) gstore16<kNt>(a + 16 * ((uint64_t)u * kWave + l), v[u]);
    } else {
        // every lane loads (vector 0 where it has none: in range, since nvec >= 1), only the
        // stores are conditional -- loads under a condition would leave every vector's
        // register live on both sides of the branch
#pragma unroll
        for (int u = 0; u < kP2pU; u++) {
            const uint64_t k = (uint64_t)u * kWave + l;
            v[u] = load(sa + 16 * (k < nvec ? k : 0));
        }
#pragma unroll
        for (int u = 0; u < kP2pU; u++) {
            const uint64_t k = (uint64_t)u * kWave + l;
            if (k < nvec) gstore16<kNt>(a + 16 * k, v[u]);
        }
    }
}

// Largest i < n with at(i) <= c (at non-decreasing, at(0) <= c); wave-uniform, 64-ary.
template <class F>
__device__ __forceinline__ int64_t p2p_search(int64_t n, uint64_t c, F at) {
    int64_t lo = 0, hi = n;
    while (hi - lo > 1) {
        const int64_t step = (hi - lo + kWave - 1) / kWave;
        const int64_t probe = lo + (int64_t)lane() * step;
        const bool le = probe < hi && at(probe < hi ? probe : lo) <= c;
        const uint64_t m = ballot(le);                 // lane 0 (probe = lo) always holds
        lo += (int64_t)(63 - __builtin_clzll(m)) * step;
        hi = lo + step < hi ? lo + step : hi;
    }
    return lo;
}

// Chunks [c0, c1), c0 in pair i; first(j) = pair j's first chunk.
template <int C, class F>
__device__ __forceinline__ void p2p_copy_chunks(const P2pPair* pairs, int64_t i, uint64_t c0, uint64_t c1, F first) {
    uint64_t here = bcast(first(i)), next = bcast(first(i + 1));
    P2pPair p = pairs[i];
    for (uint64_t c = c0; c < c1; c++) {
        if (c >= next) {
            do {                                             // skips empty pairs
                here = next;
                next = bcast(first(++i + 1));
            } while (c >= next);
            p = pairs[i];
        }
        const uint64_t d = (uint64_t)(uintptr_t)p.dst;
        const uint64_t blk = ((d >> kP2pChunkShift) + (c - here)) << kP2pChunkShift;
        const uint64_t plo = blk > d ? blk : d;
        const uint64_t phi = blk + kP2pChunk < d + p.bytes ? blk + kP2pChunk : d + p.bytes;
        p2p_copy_piece<C>(p.dst, p.src, plo, phi);
    }
}

// The copy, by workgroups of NT threads.  FUSED: n <= FUSED pairs and no scan kernel ran; s_off
// holds every pair's first chunk.  FUSED = 0: s_off holds every tile's first chunk, and a pair's
// is its tile's plus chunk_off.
template <int FUSED, int NT, int WAVES>
static __global__ __launch_bounds__(NT, WAVES) void p2p_copy_kernel(const P2pPair* pairs, int64_t n, int tile_shift,
                                                             const uint64_t* chunk_off, const uint64_t* tile_chunks) {
    __shared__ uint64_t s_off[FUSED ? FUSED : kP2pTiles];
    __shared__ uint64_t s_w[NT / kWave];
    const int64_t tiles = FUSED ? n : (n + (1ll << tile_shift) - 1) >> tile_shift;
    uint64_t total;
    if constexpr (FUSED != 0) {
        total = p2p_scan_pass<NT, FUSED>(pairs, 0, n, 0, s_off, s_w);
    } else {
        constexpr int kPer = kP2pTiles / NT;
        uint64_t c[kPer], sum = 0;
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int b = (int)threadIdx.x * kPer + k;
            c[k] = b < tiles ? tile_chunks[b] : 0;
            sum += c[k];
        }
        uint64_t run = p2p_block_scan<NT>(sum, s_w, &total);
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            s_off[threadIdx.x * kPer + k] = run;
            run += c[k];
        }
        __syncthreads();
    }
    // first chunk of pair i, i <= n
    auto first = [&](int64_t i) -> uint64_t {
        if (i >= n) return total;
        if constexpr (FUSED != 0) return s_off[i];
        else return s_off[i >> tile_shift] + chunk_off[i];
    };
    const uint64_t nw = (uint64_t)gridDim.x * (NT / kWave);
    // the wave index through readfirstlane: everything derived from it (the chunk range,
    // the search, the pair fields) is then wave-uniform and kept in SGPRs
    const uint64_t w = (uint64_t)blockIdx.x * (NT / kWave) + bcast((uint32_t)(threadIdx.x >> 6));
    const uint64_t c0 = total * w / nw, c1 = total * (w + 1) / nw;
    if (c0 >= c1) return;
    int64_t i = p2p_search(tiles, c0, [&](int64_t k) { return s_off[k]; });
    if constexpr (FUSED == 0) {
        const int64_t b = i << tile_shift, left = n - b;
        const uint64_t in_tile = c0 - bcast(s_off[i]);
        i = b + p2p_search(left < (1ll << tile_shift) ? left : 1ll << tile_shift, in_tile,
                           [&](int64_t k) { return chunk_off[b + k]; });
    }
    // a loop each: with the choice at each store, the compiler makes one cached store of both kinds
    const P2pCaching kind = p2p_caching(bcast(total), n);
    if (kind == kP2pCached) p2p_copy_chunks<kP2pCached>(pairs, i, c0, c1, first);
    else if (kind == kP2pKeepStores) p2p_copy_chunks<kP2pKeepStores>(pairs, i, c0, c1, first);
    else p2p_copy_chunks<kP2pKeepNothing>(pairs, i, c0, c1, first);
}

}  // namespace gpumpi
