// Batched MPI_Alltoallv step: a plan, a scan and a copy kernel (plan and scan in one for up to 64
// ranks; in pipelined graphs the copy plans the next step), replayed from hipGraphs.
//
// Semantics: gpu_mpi/mpi.cu:363-408 (block s of rank d's receive buffer <- block d of
// rank s's send buffer, counts/displacements in elements), preceded by the Alltoall of
// the counts and the packed receive displacements that the NPB IS caller computes
// between the two calls (toolchain_tests/npb/NPB3.4.1/NPB3.4-MPI/IS/is.c:758-781).
//
// The reference runs this as P-1 Isend + P-1 Irecv per rank, each payload copied by one
// thread.  Here the step is decoupled from ranks and split at the only global dependency
// (the receive displacements need every sender's count):
//
//  plan   one workgroup per destination row d: recv_counts[d][s] = send_counts[s][d],
//         recv_displs = exclusive scan over s, and per segment (d, s) its end offset in
//         the row and its source address.
//  scan   one workgroup: chunks per row (a row's destination lines, counted from the
//         128-byte block holding its first byte, cut into chunks of chunk_lines 16-byte
//         lines) and their exclusive prefix.
//  copy   one workgroup per chunk (grid-stride when the grid is smaller): wave 0 finds
//         the chunk's row and first segment (64-ary searches over L2-resident tables)
//         and stages a window of 64 segments in LDS; each wave then copies a contiguous
//         run of 64*U lines slice by slice, keeping a wave-uniform cursor into the window
//         (it only moves forward; kept in SGPRs) and, when the slice does not lie in one
//         entry, choosing each lane's segment among the cursor's next four with compares.
//         The loop is bound by instruction issue, so the common cases are uniform paths:
//         a slice inside one segment costs one source offset from SGPRs, a slice across
//         one boundary a per-lane choice between two.  A line inside one segment is
//         one unaligned 16-byte load and one aligned 16-byte store; a line that straddles
//         segments is four dword loads (issued with the other lines' loads) and one
//         16-byte store -- or, in
//         deferred mode (a tuning choice that pays when segments are short, as in skewed
//         key distributions), left to one thread per segment run by the grid's first
//         blocks, concurrently with the streaming blocks.  Dwords that are split or unaligned
//         at the source go byte by byte; bytes outside the row are never written.  The lines
//         at the ends of rows are a lane each in the first blocks.
//         Rows of short segments, of elements that are not whole dwords, and small rows take
//         a loop of their own (a2av_copy_short), in which each lane finds its line's segments.
//         Measured (execute, us, before -> with it): 16 ranks x 3 KiB 24.0 -> 12.9 (11.2 since
//         up to 64 ranks are planned and scanned by one kernel and their tables read in one
//         round); 200 ranks, 48 MiB of bytes, segments of 157 B to 50 KiB 403 -> 39; 512 ranks,
//         64-byte segments, 16 MiB 95 -> 35.
//
// Why not one persistent kernel with a grid barrier: on gfx950 an agent-scope release or
// acquire writes back or invalidates the XCD's L2 (buffer_wbl2 / buffer_inv sc1); a grid
// barrier across 256-2048 workgroups measured 14-150 us, a kernel boundary inside a graph
// a few us.  And a copy grid of many short workgroups streams faster than a persistent
// grid (5.9 vs 5.0-5.2 TB/s for a plain 512 MiB copy on MI355X).
//
// HBM traffic per step = payload read once + payload written once + O(P^2) tables
// (counts and displacements read, 4 + 4 + 8 + 8 bytes per segment written and read).
#pragma once

#include "copy.h"

namespace gpumpi {

constexpr int kA2avWindow = 64;
constexpr int kA2avCopyThreads = 256;

// Short rows are copied line by line (a2av_copy_short): every lane finds its own line's
// segments.  Their chunks are smaller, so that more workgroups share them.  A row is short
// when its non-empty segments average less than kA2avShortBytes (kA2avShortOdd if the elements
// are not whole dwords, which the other loop assembles byte by byte at every boundary), or when
// it is too small to be a stream at all.  Where the lines lie, measured (short / long loop, us):
// 256 ranks of dwords, segments of 256 B 24.9 / 38.7, 512 B 33.6 / 32.3, 1 KiB 49 / 38; of
// bytes, 4 KiB 147 / 257, 16 KiB 516 / 706, 64 KiB (32 ranks) 39 / 37; 4 ranks x 4 KiB rows
// 13.3 / 15.4, 8 KiB 12.6 / 13.0, 16 KiB 13.6 / 12.8.
constexpr uint64_t kA2avShortRow = 1ull << 63;
constexpr uint64_t kA2avShortBytes = 448;
constexpr uint64_t kA2avShortOdd = 32768;
constexpr uint64_t kA2avSmallRow = 8192;
// Lines per chunk of a short row: 16 KiB, up to 64 KiB in steps that give twice kA2avChunks of
// them (finding a chunk's row and segments takes about as long as copying 16 KiB).
constexpr uint64_t kA2avShortLines = 1024, kA2avShortMost = 4096;
constexpr int kA2avShortWindow = 512;
constexpr uint64_t kA2avChunks = 2048;    // chunks that keep the chip busy

struct A2avDev {
    int32_t P;
    int32_t elem;
    uint32_t chunk_lines;   // destination lines per chunk at most: kA2avCopyThreads * U * rounds
    uint32_t min_lines;     // and at least: kA2avCopyThreads * U
    int32_t straddle_blocks;  // deferred mode: leading copy blocks running the straddle threads
    char* const* sendbufs;
    const int32_t* scounts;
    const int32_t* sdispls;
    char* const* recvbufs;
    int32_t* rcounts;
    int32_t* rdispls;
    uint64_t* seg_end;      // [P*P] end byte offset of segment (d, s) within row d
    uint64_t* seg_src;      // [P*P] address of the first source byte of segment (d, s)
    uint64_t* row_bytes;    // [P], with kA2avShortRow set in rows of short segments
    uint64_t* chunk_off;    // [P+1] exclusive prefix of chunks per long row; [P] = all of them
    uint64_t* short_off;    // [P+1] the same for the short rows
    int64_t* total_bytes;   // [0] payload; [1] lines per chunk of the long rows, [2] of the short
    uint32_t* plan_done;    // [1] plan workgroups finished (fused plan; reset by the last one)
};

__device__ __forceinline__ int64_t wave_excl_scan(int64_t v, int64_t* total) {
    int64_t inc = wave_incl_scan(v);
    *total = __shfl(inc, 63);
    return inc - v;
}

// Largest i in [0, n) with a[i] <= x (a non-decreasing, a[0] <= x); wave-uniform,
// 64-ary: each step compares 64 evenly spaced entries.
__device__ __forceinline__ int64_t wave_search_le(const uint64_t* a, int64_t n, uint64_t x) {
    int64_t lo = 0, hi = n;
    while (hi - lo > 1) {
        const int64_t step = (hi - lo + 63) / 64;
        const int64_t idx = lo + (int64_t)lane() * step;
        const bool le = idx < hi && a[idx] <= x;
        const uint64_t m = ballot(le);
        const int L = m ? 63 - __builtin_clzll(m) : 0;
        const int64_t nlo = lo + (int64_t)L * step;
        const int64_t nhi = nlo + step;
        lo = nlo;
        hi = nhi < hi ? nhi : hi;
    }
    return lo;
}

// A row's byte count, marked if the row is short (deferred mode has its own way with short
// segments).
__device__ __forceinline__ uint64_t a2av_row_word(const A2avDev& p, uint64_t bytes, uint64_t nonempty) {
    const bool small = bytes < kA2avSmallRow || bytes < nonempty * (p.elem & 3 ? kA2avShortOdd : kA2avShortBytes);
    return p.straddle_blocks == 0 && small ? bytes | kA2avShortRow : bytes;
}

// ------------------------------------------------------------------------------ plan
// One workgroup of four wavefronts per destination row d; wave w owns a contiguous
// quarter of the sources.  The first 256 sources of a quarter (all of them up to P = 1024)
// are loaded once -- counts, displacements and send buffers in one round of loads -- and
// kept in registers: the quarters' count totals meet in LDS to give each quarter's
// starting displacement, then each wave scans and writes.  Sources past 256 per quarter
// are summed in a first pass and reloaded in the second.
// COHERENT: the row's byte count is stored with an agent-scope atomic store (written
// through to memory), for a reader in the same kernel on another XCD.
template <bool COHERENT = false>
__device__ __forceinline__ void a2av_plan_row(const A2avDev& p, int64_t d, int64_t* s_tot) {
    const int P = p.P;
    const int l = lane();
    const int w = threadIdx.x >> 6;
    const int Q = (((P + 3) / 4) + kWave - 1) / kWave * kWave;
    const int sb = w * Q;
    const int se = sb + Q < P ? sb + Q : P;
    int64_t c[4], sd[4];
    const char* sbuf[4];
    int64_t part = 0;        // elements, and non-empty segments from bit 44 on
    constexpr int kSegShift = 44;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int s = sb + q * kWave + l;
        const bool valid = s < se;
        c[q] = valid ? p.scounts[(int64_t)s * P + d] : 0;
        sd[q] = valid ? p.sdispls[(int64_t)s * P + d] : 0;
        sbuf[q] = valid ? p.sendbufs[s] : nullptr;
        part += c[q] + (c[q] > 0 ? 1ll << kSegShift : 0);
    }
    for (int s0 = sb + 4 * kWave; s0 < se; s0 += kWave) {
        const int s = s0 + l;
        const int64_t x = s < se ? p.scounts[(int64_t)s * P + d] : 0;
        part += x + (x > 0 ? 1ll << kSegShift : 0);
    }
    part = wave_sum(part);
    if (l == 0) s_tot[w] = part;
    __syncthreads();
    int64_t carry = 0, row = 0, nonempty = 0;
    for (int k = 0; k < 4; k++) {
        const int64_t x = s_tot[k] & ((1ll << kSegShift) - 1);
        carry += k < w ? x : 0;
        row += x;
        nonempty += s_tot[k] >> kSegShift;
    }
    for (int s0 = sb; s0 < se; s0 += kWave) {
        const int q = (s0 - sb) / kWave;
        const int s = s0 + l;
        int64_t cq, sdq;
        const char* sbq;
        if (q < 4) {
            cq = q == 0 ? c[0] : q == 1 ? c[1] : q == 2 ? c[2] : c[3];
            sdq = q == 0 ? sd[0] : q == 1 ? sd[1] : q == 2 ? sd[2] : sd[3];
            sbq = q == 0 ? sbuf[0] : q == 1 ? sbuf[1] : q == 2 ? sbuf[2] : sbuf[3];
        } else {
            const bool valid = s < se;
            cq = valid ? p.scounts[(int64_t)s * P + d] : 0;
            sdq = valid ? p.sdispls[(int64_t)s * P + d] : 0;
            sbq = valid ? p.sendbufs[s] : nullptr;
        }
        int64_t tot;
        const int64_t rd = wave_excl_scan(cq, &tot) + carry;
        carry += tot;
        if (s < se) {
            const int64_t o = d * P + s;
            p.rcounts[o] = (int32_t)cq;
            p.rdispls[o] = (int32_t)rd;
            p.seg_end[o] = (uint64_t)(rd + cq) * (uint64_t)p.elem;
            p.seg_src[o] = (uint64_t)(uintptr_t)(sbq + sdq * p.elem);
        }
    }
    if (threadIdx.x == 0) {
        const uint64_t rb = a2av_row_word(p, (uint64_t)row * (uint64_t)p.elem, (uint64_t)nonempty);
        if constexpr (COHERENT) st_relaxed(&p.row_bytes[d], rb);
        else p.row_bytes[d] = rb;
    }
}

static __global__ void __launch_bounds__(256) a2av_plan_kernel(A2avDev p) {
    __shared__ int64_t s_tot[4];
    a2av_plan_row(p, blockIdx.x, s_tot);
}

// ------------------------------------------------------------------------------ scan
// Run by one workgroup of NT threads (NT a multiple of 64, at most 1024).  COHERENT: the
// row byte counts are read with agent-scope atomic loads (written in the same kernel).
template <int NT, bool COHERENT = false>
__device__ __forceinline__ void a2av_scan_rows(const A2avDev& p, uint64_t* part, int64_t* bpart) {
    constexpr int NW = NT / kWave;
    const int P = p.P;
    const int w = threadIdx.x >> 6;
    auto row_word = [&](int d) { return COHERENT ? ld_relaxed(&p.row_bytes[d]) : p.row_bytes[d]; };
    int64_t bytes = 0;
    for (int base = 0; base < P; base += NT) {
        const int d = base + (int)threadIdx.x;
        bytes += d < P ? (int64_t)(row_word(d) & ~kA2avShortRow) : 0;
    }
    bytes = wave_sum(bytes);
    if (lane() == 0) bpart[w] = bytes;
    __syncthreads();
    bytes = 0;
    for (int k = 0; k < NW; k++) bytes += bpart[k];
    // smaller chunks while the payload does not give kA2avChunks of them
    uint64_t C = p.chunk_lines;
    while (C > p.min_lines && (uint64_t)bytes / 16 < C * kA2avChunks) C >>= 1;
    uint64_t S = kA2avShortMost;
    while (S > kA2avShortLines && (uint64_t)bytes / 16 < S * 2 * kA2avChunks) S >>= 1;
    uint64_t carry = 0;      // chunks of long rows, and of short rows from bit 32 on
    for (int base = 0; base < P; base += NT) {
        const int d = base + (int)threadIdx.x;
        uint64_t ch = 0;
        if (d < P) {
            const uint64_t word = row_word(d), nb = word & ~kA2avShortRow;
            const uint64_t rb = (uint64_t)(uintptr_t)p.recvbufs[d];
            const uint64_t lines = nb ? ((rb + nb + 15) >> 4) - ((rb >> 7) << 3) : 0;
            ch = word & kA2avShortRow ? ((lines + S - 1) / S) << 32 : (lines + C - 1) / C;
        }
        const uint64_t inc = (uint64_t)wave_incl_scan((int64_t)ch);
        if (lane() == 63) part[w] = inc;
        __syncthreads();
        uint64_t before = 0, total = 0;
        for (int k = 0; k < NW; k++) {
            if (k < w) before += part[k];
            total += part[k];
        }
        if (d < P) {
            const uint64_t off = carry + before + inc - ch;
            p.chunk_off[d] = (uint32_t)off;
            p.short_off[d] = off >> 32;
        }
        carry += total;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        p.chunk_off[P] = (uint32_t)carry;
        p.short_off[P] = carry >> 32;
        p.total_bytes[0] = bytes;
        p.total_bytes[1] = (int64_t)C;
        p.total_bytes[2] = (int64_t)S;
    }
}

static __global__ void __launch_bounds__(1024) a2av_scan_kernel(A2avDev p) {
    __shared__ uint64_t part[16];
    __shared__ int64_t bpart[16];
    a2av_scan_rows<1024>(p, part, bpart);
}

// Plan and scan of at most 64 ranks by one workgroup: a wave per row, a lane per source.  One
// launch less per step (16 ranks x 3 KiB 12.9 -> 11.8 us); more ranks need the plan's P
// workgroups.
constexpr int kA2avSmallRanks = 64;
static __global__ void __launch_bounds__(1024) a2av_plan_small_kernel(A2avDev p) {
    __shared__ uint64_t part[16];
    __shared__ int64_t bpart[16];
    const int P = p.P, l = lane();
    for (int d = threadIdx.x >> 6; d < P; d += 16) {
        const bool valid = l < P;
        const int s = valid ? l : 0;
        const int64_t c = valid ? p.scounts[(int64_t)s * P + d] : 0;
        const int64_t sd = p.sdispls[(int64_t)s * P + d];
        const char* sbuf = p.sendbufs[s];
        int64_t tot;
        const int64_t rd = wave_excl_scan(c, &tot);
        const uint32_t nonempty = (uint32_t)__popcll(ballot(c > 0));
        if (valid) {
            const int64_t o = (int64_t)d * P + s;
            p.rcounts[o] = (int32_t)c;
            p.rdispls[o] = (int32_t)rd;
            p.seg_end[o] = (uint64_t)(rd + c) * (uint64_t)p.elem;
            p.seg_src[o] = (uint64_t)(uintptr_t)(sbuf + sd * p.elem);
        }
        if (l == 0) p.row_bytes[d] = a2av_row_word(p, (uint64_t)tot * (uint64_t)p.elem, nonempty);
    }
    __syncthreads();
    a2av_scan_rows<1024>(p, part, bpart);
}

// Plan of the NEXT step run by the first P workgroups of a copy kernel (the step's only
// global dependency -- the receive displacements -- is then resolved while the current
// step streams, instead of in kernels of its own on the critical path).  The tables go to
// the other of two workspaces, so the copy running beside them is not disturbed.
//
// With pn.plan_done set, the workgroup that finishes last also computes the chunk prefix.
// Only the row byte counts cross workgroups inside the kernel (everything else is read by
// the next kernel): each planner stores its count with an agent-scope atomic store, which
// writes through to memory, waits for that store to complete, then counts itself done;
// the last one reads the counts with agent-scope atomic loads, which miss the L2.  No L2
// write-back or invalidate is needed (agent-scope fences in 512 workgroups, writing back
// their XCDs' L2s under the streaming copy, cost 35-60 us per step).
// With pn.plan_done == nullptr the workgroups only plan; a scan kernel follows.
__device__ void a2av_plan_fused(const A2avDev& pn, int64_t d) {
    __shared__ int64_t s_tot[4];
    __shared__ uint64_t s_part[4];
    __shared__ int64_t s_bpart[4];
    __shared__ int32_t s_last;
    if (!pn.plan_done) {  // block-uniform
        a2av_plan_row<false>(pn, d, s_tot);
        return;
    }
    a2av_plan_row<true>(pn, d, s_tot);
    if (threadIdx.x == 0) {
        wait_mem_done();
        const uint32_t old = __hip_atomic_fetch_add(pn.plan_done, 1u, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
        s_last = old == (uint32_t)pn.P - 1u;
    }
    __syncthreads();
    if (!s_last) return;
    a2av_scan_rows<kA2avCopyThreads, true>(pn, s_part, s_bpart);
    if (threadIdx.x == 0) *pn.plan_done = 0u;  // next used two kernels later
}

// ------------------------------------------------------------------------------ straddle
// Deferred mode: lines inside a row that hold bytes of two or more segments.  One thread
// per segment of every row; a segment whose end falls strictly inside a 16-byte line, and
// that holds that line's first byte, owns the line: it assembles it per dword from the
// segment holding each dword (per byte where a dword is split or unaligned at its source)
// and stores it once.  Every such line has exactly one owner.  Lines across a row's ends
// stay with the copy loop.  The copy grid's first straddle_blocks blocks run these
// threads: their scattered, latency-bound loads overlap the other blocks' streaming.
__device__ void a2av_straddle_line(const A2avDev& p, uint64_t gid) {
    const int P = p.P;
    if (gid >= (uint64_t)P * (uint64_t)P) return;
    const int64_t d = (int64_t)(gid / (uint64_t)P);
    const int s = (int)(gid - (uint64_t)d * P);
    const uint64_t* se = p.seg_end + d * P;
    // one round of independent loads: this segment, the next one, the row
    const int s1 = s + 1 < P ? s + 1 : s;
    const int64_t prev = (int64_t)se[s > 0 ? s - 1 : 0];
    const int64_t en = (int64_t)se[s];
    const int64_t en1 = (int64_t)se[s1];
    const uint64_t src0 = p.seg_src[d * P + s];
    const uint64_t src1 = p.seg_src[d * P + s1];
    const uint64_t rbase = (uint64_t)(uintptr_t)p.recvbufs[d];
    const int64_t rbytes = (int64_t)(p.row_bytes[d] & ~kA2avShortRow);
    const int64_t st = s > 0 ? prev : 0;
    if (en <= st) return;  // empty
    const uint64_t le = rbase + (uint64_t)en;  // one past the segment's last byte
    if ((le & 15) == 0) return;                // ends with its line
    const uint64_t la = (le >> 4) << 4;        // the line holding the segment's last byte
    const int64_t off = (int64_t)la - (int64_t)rbase;
    if (st > off || off < 0 || off + 16 > rbytes) return;
    // the next non-empty segment
    int kb = s + 1;
    int64_t eb = en1;
    uint64_t srcb = src1;
    if (en1 <= en) {
        while ((int64_t)se[kb] <= en) kb++;  // ends before rbytes >= off + 16 > en
        eb = (int64_t)se[kb];
        srcb = p.seg_src[d * P + kb];
    }
    const uint64_t a0 = src0 + (uint64_t)(off - st);  // source of the line's byte 0 in s
    const uint64_t a1 = srcb - (uint64_t)en;          // + row offset, in segment kb
    if (eb >= off + 16) {
        // two segments: four loads in flight
        uint64_t addr[4];
        bool whole[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t q = off + 4 * i;
            const bool first = q < en;
            addr[i] = first ? a0 + 4 * i : a1 + (uint64_t)q;
            whole[i] = (!first || q + 4 <= en) && (addr[i] & 3) == 0;
        }
        uint32_t v[4];
        // a dword split between the segments, or unaligned at its source, is fetched per
        // byte; its aligned-down dword holds a byte of the source and is a safe read
#pragma unroll
        for (int i = 0; i < 4; i++)
            v[i] = *(const GPUMPI_GLOBAL uint32_t*)(uintptr_t)(addr[i] & ~(uint64_t)3);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (whole[i]) continue;
            uint32_t x = 0;
            for (int j = 0; j < 4; j++) {
                const int64_t b = off + 4 * i + j;
                const uint64_t ab = b < en ? a0 + 4 * i + j : a1 + (uint64_t)b;
                x |= (uint32_t)*(const GPUMPI_GLOBAL uint8_t*)(uintptr_t)ab << (8 * j);
            }
            v[i] = x;
        }
        *(GPUMPI_GLOBAL u32x4*)(uintptr_t)la = u32x4{v[0], v[1], v[2], v[3]};
        return;
    }
    // three or more segments in the line: walk them
    int k = s;  // holds byte `off`; the walk only moves forward over the line
    uint64_t src[4];
    int whole = 0;
    for (int i = 0; i < 4; i++) {
        const int64_t q = off + 4 * i;
        while (q >= (int64_t)se[k]) k++;
        const int64_t sk = k > 0 ? (int64_t)se[k - 1] : 0;
        src[i] = p.seg_src[d * P + k] + (uint64_t)(q - sk);
        if (q + 4 <= (int64_t)se[k] && (src[i] & 3) == 0) whole |= 1 << i;
    }
    uint32_t v[4];
    k = s;
    for (int i = 0; i < 4; i++) {
        if (whole & (1 << i)) {
            v[i] = *(const GPUMPI_GLOBAL uint32_t*)(uintptr_t)src[i];
            continue;
        }
        uint32_t x = 0;
        for (int j = 0; j < 4; j++) {
            const int64_t b = off + 4 * i + j;
            while (b >= (int64_t)se[k]) k++;
            const int64_t sb = k > 0 ? (int64_t)se[k - 1] : 0;
            const uint8_t y = *(const GPUMPI_GLOBAL uint8_t*)(uintptr_t)(p.seg_src[d * P + k] +
                                                                        (uint64_t)(b - sb));
            x |= (uint32_t)y << (8 * j);
        }
        v[i] = x;
    }
    *(GPUMPI_GLOBAL u32x4*)(uintptr_t)la = u32x4{v[0], v[1], v[2], v[3]};
}

// ------------------------------------------------------------------------------ copy
// One segment seen from its row: bytes [st, en) of the row; the source of the row byte at
// offset q is (rbase + q) + D.
struct A2avSegView {
    int64_t st, en;
    uint64_t D;
};

// Segment holding row offset q (0 <= q < row bytes), by binary search over the row's
// segment ends in HBM (the path for lines outside the LDS window).
__host__ __device__ __forceinline__ A2avSegView a2av_seg_global(const A2avDev& p, int64_t d, uint64_t rbase,
                                                       int64_t q) {
    const uint64_t* se = p.seg_end + d * p.P;
    int64_t lo = 0, hi = p.P - 1;  // first s with se[s] > q
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)se[mid] > q) hi = mid; else lo = mid + 1;
    }
    A2avSegView v;
    v.st = lo > 0 ? (int64_t)se[lo - 1] : 0;
    v.en = (int64_t)se[lo];
    v.D = p.seg_src[d * p.P + lo] - (rbase + (uint64_t)v.st);
    return v;
}

// Window entry holding row offset q (s_st[0] <= q < coverage): largest k < cnt with
// s_st[k] <= q.  cnt is wave-uniform, so the search takes ceil(log2(cnt)) steps.
__device__ __forceinline__ int a2av_seg_lds(const int64_t* s_st, int cnt, int64_t q) {
    int k = 0;
    for (int b = cnt > 1 ? 1 << (31 - __builtin_clz(cnt - 1)) : 0; b > 0; b >>= 1)
        if (k + b < cnt && s_st[k + b] <= q) k += b;
    return k;
}

struct A2avWin {
    const int64_t* st;
    const int64_t* en;
    const uint64_t* D;
    int cnt;
    int nsearch;        // entries starting before the pass's last line: the search range
    int64_t lo, cover;  // row offsets [lo, cover) are described by the window
};

__device__ __forceinline__ A2avSegView a2av_seg_at(const A2avDev& p, int64_t d, uint64_t rbase,
                                                   const A2avWin& w, int64_t q) {
    if (q >= w.lo && q < w.cover) {
        const int k = a2av_seg_lds(w.st, w.nsearch, q);
        return A2avSegView{w.st[k], w.en[k], w.D[k]};
    }
    return a2av_seg_global(p, d, rbase, q);
}

// Bytes at .. at + 3 (at & 3) of the 8 bytes lo, hi.
__host__ __device__ __forceinline__ uint32_t byte_funnel(uint32_t hi, uint32_t lo, uint32_t at) {
#ifdef __HIP_DEVICE_COMPILE__
    return (uint32_t)__builtin_amdgcn_alignbyte(hi, lo, at);
#else
    return (uint32_t)(((uint64_t)hi << 32 | lo) >> (8 * (at & 3)));
#endif
}

// 16 bytes from byte `at` (0..16) of the 32 bytes a, b.
__host__ __device__ __forceinline__ u32x4 bytes_from(u32x4 a, u32x4 b, uint32_t at) {
    const bool h16 = at & 16, h8 = at & 8, h4 = at & 4;
    // (scalars: an array would be indexed in scratch memory)
    uint32_t x0 = h16 ? b.x : a.x, x1 = h16 ? b.y : a.y, x2 = h16 ? b.z : a.z, x3 = h16 ? b.w : a.w;
    uint32_t x4 = b.x, x5 = b.y, x6 = b.z;       // (past byte 16 nothing follows)
    x0 = h8 ? x2 : x0;
    x1 = h8 ? x3 : x1;
    x2 = h8 ? x4 : x2;
    x3 = h8 ? x5 : x3;
    x4 = h8 ? x6 : x4;
    x5 = h8 ? b.w : x5;
    x0 = h4 ? x1 : x0;
    x1 = h4 ? x2 : x1;
    x2 = h4 ? x3 : x2;
    x3 = h4 ? x4 : x3;
    x4 = h4 ? x5 : x4;
    return u32x4{byte_funnel(x1, x0, at), byte_funnel(x2, x1, at), byte_funnel(x3, x2, at), byte_funnel(x4, x3, at)};
}

// Bytes [0, n) at address a, n < 16, in the low bytes; reads nothing else.
__host__ __device__ __forceinline__ u32x4 load_bytes(uint64_t a, uint32_t n) {
    typedef uint64_t u64_a1 __attribute__((aligned(1)));
    typedef uint32_t u32_a1 __attribute__((aligned(1)));
    typedef uint16_t u16_a1 __attribute__((aligned(1)));
    uint64_t lo = 0, r = 0;
    uint32_t f = 0, g = 0;
    if (n & 8) {
        lo = *(const GPUMPI_GLOBAL u64_a1*)(uintptr_t)a;
        f = 8;
    }
    if (n & 4) {
        r = *(const GPUMPI_GLOBAL u32_a1*)(uintptr_t)(a + f);
        g = 4;
    }
    if (n & 2) {
        r |= (uint64_t)*(const GPUMPI_GLOBAL u16_a1*)(uintptr_t)(a + f + g) << (8 * g);
        g += 2;
    }
    if (n & 1) r |= (uint64_t)*(const GPUMPI_GLOBAL uint8_t*)(uintptr_t)(a + f + g) << (8 * g);
    if (!(n & 8)) { lo = r; r = 0; }
    return u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)r, (uint32_t)(r >> 32)};
}

// The destination line `line` of a row, from however many segments it holds: at(q) is the
// segment holding row byte q.  Each piece is one 16-byte load from inside its segment, moved to
// its bytes (a segment of less than 16 bytes: up to four smaller loads); only row bytes are
// read and written.  A byte at a time -- a search, a load and a store for each of 16 -- such lines took
// most of a copy of short unaligned segments.
template <class F>
__host__ __device__ __forceinline__ void a2av_assemble_line(uint64_t rbase, int64_t rbytes, uint64_t line, F at) {
    const uint64_t la = line << 4;
    const int64_t off = (int64_t)la - (int64_t)rbase;
    const int b0 = off >= 0 ? 0 : off <= -16 ? 16 : (int)-off;
    const int b1 = rbytes - off >= 16 ? 16 : (int)(rbytes - off);
    if (b0 >= b1) return;
    uint32_t acc[4] = {0, 0, 0, 0};
    for (int pos = b0; pos < b1;) {
        const A2avSegView sg = at(off + pos);
        const int64_t end = sg.en - off, start = sg.st - off;      // in line bytes
        const int e = end < b1 ? (int)end : b1;
        const uint64_t src = la + sg.D;                            // of line byte 0
        const u32x4 none{0u, 0u, 0u, 0u};
        u32x4 y;
        if (end - start >= 16) {
            int64_t f = start > 0 ? start : 0;
            if (f > end - 16) f = end - 16;                        // -15 .. 15
            const u32x4 x = gload16(src + (uint64_t)f);
            y = bytes_from(f >= 0 ? none : x, f >= 0 ? x : none, (uint32_t)(f >= 0 ? 16 - f : -f));
        } else {
            y = bytes_from(none, load_bytes(src + (uint64_t)pos, (uint32_t)(e - pos)), 16u - (uint32_t)pos);
        }
        const uint32_t w[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int a = pos - 4 * i, b = e - 4 * i;
            const uint64_t upto = (1ull << (8 * (b < 0 ? 0 : b > 4 ? 4 : b))) - 1;
            const uint64_t skip = (1ull << (8 * (a < 0 ? 0 : a > 4 ? 4 : a))) - 1;
            acc[i] |= w[i] & (uint32_t)(upto & ~skip);
        }
        pos = e;
    }
    if (b0 == 0 && b1 == 16) {
        *(GPUMPI_GLOBAL u32x4*)(uintptr_t)la = u32x4{acc[0], acc[1], acc[2], acc[3]};
        return;
    }
    for (int b = b0; b < b1; b++) {
        const uint32_t x = b < 4 ? acc[0] : b < 8 ? acc[1] : b < 12 ? acc[2] : acc[3];
        *(GPUMPI_GLOBAL uint8_t*)(uintptr_t)(la + b) = (uint8_t)(x >> (8 * (b & 3)));
    }
}

// A destination line that straddles segments (deferred mode, whose straddle threads have
// those: the row's ends): assembled per dword (per byte where a dword is split or its source
// unaligned); only row bytes are written.
template <bool DEFER>
__device__ void a2av_boundary_line(const A2avDev& p, int64_t d, uint64_t rbase, int64_t rbytes,
                                   const A2avWin& w, uint64_t line) {
    const uint64_t la = line << 4;
    const int64_t off = (int64_t)la - (int64_t)rbase;
    // deferred mode: only the lines at the row's ends are left; otherwise only those inside it
    if (DEFER == (off >= 0 && off + 16 <= rbytes)) return;
    uint32_t v[4] = {0, 0, 0, 0};
    int mask = 0;
    for (int i = 0; i < 4; i++) {
        const int64_t q = off + 4 * i;
        if (q >= 0 && q + 4 <= rbytes) {
            const A2avSegView sg = a2av_seg_at(p, d, rbase, w, q);
            const uint64_t src = la + 4 * i + sg.D;
            if (q + 4 <= sg.en && (src & 3) == 0) {
                v[i] = *(const GPUMPI_GLOBAL uint32_t*)(uintptr_t)src;
                mask |= 1 << i;
                continue;
            }
        }
        for (int j = 0; j < 4; j++) {
            const int64_t b = q + j;
            if (b < 0 || b >= rbytes) continue;
            const A2avSegView sg = a2av_seg_at(p, d, rbase, w, b);
            const uint64_t a = la + 4 * i + j;
            *(GPUMPI_GLOBAL uint8_t*)(uintptr_t)a = *(const GPUMPI_GLOBAL uint8_t*)(uintptr_t)(a + sg.D);
        }
    }
    if (mask == 0xF) {
        *(GPUMPI_GLOBAL u32x4*)(uintptr_t)la = u32x4{v[0], v[1], v[2], v[3]};
    } else {
        for (int i = 0; i < 4; i++)
            if (mask & (1 << i)) *(GPUMPI_GLOBAL uint32_t*)(uintptr_t)(la + 4 * i) = v[i];
    }
}

// The first (which = 0) or last line of long row d, if it holds bytes of the row and others.
// (Left to the copy loop, whose lane assembles it byte by byte, such a line holds up the
// workgroup that ends its row by some 20 us.)
__host__ __device__ __forceinline__ void a2av_row_end(const A2avDev& p, int64_t d, int which) {
    const uint64_t word = p.row_bytes[d];
    if (word == 0 || (word & kA2avShortRow)) return;
    const uint64_t rbase = (uint64_t)(uintptr_t)p.recvbufs[d], rend = rbase + word;
    if (((which ? rend : rbase) & 15) == 0) return;
    const uint64_t first = rbase >> 4, last = rend >> 4;
    if (which && first == last && (rbase & 15)) return;     // one line: the first
    a2av_assemble_line(rbase, (int64_t)word, which ? last : first,
                       [&](int64_t q) { return a2av_seg_global(p, d, rbase, q); });
}

// The threads of a workgroup, as a2av_copy_short uses them (a test on the CPU runs them one after
// the other).
struct A2avGroup {
    // f by every thread, then a barrier
    template <class F>
    static __device__ __forceinline__ void each(F f) {
        f((int)threadIdx.x);
        __syncthreads();
    }
    static __device__ __forceinline__ int32_t uniform(int32_t v) { return bcast(v); }
    static __device__ __forceinline__ int64_t uniform(int64_t v) { return bcast(v); }
    // first of the n entries of se that is above o; `slot` in LDS
    static __device__ __forceinline__ int64_t first_above(const uint64_t* se, int64_t n, int64_t o, int64_t* slot) {
        each([&](int tid) {
            if (tid < kWave) {
                int64_t s0 = 0;
                if ((int64_t)se[0] <= o) s0 = wave_search_le(se, n, (uint64_t)o) + 1;
                if (tid == 0) *slot = s0;
            }
        });
        return bcast(*slot);
    }
};

// Lines [pos, line1) of a row of short segments, by the whole workgroup.  Windows of up
// to 512 segments in LDS (offsets relative to the window's first row byte `o`); each lane finds the
// segment of its line by bisection, two lines at a time, so that the searches' LDS reads and
// the lines' loads overlap.  A line across one boundary takes the 16 bytes up to the
// boundary and the 16 from it, and a funnel shift; other lines are assembled piece by piece.
// A wave-uniform cursor over the segments (the loop for long segments) gains nothing when
// every slice of 64 lines crosses several.
template <bool NT, class Group>
__host__ __device__ __forceinline__ void a2av_copy_short(const A2avDev& p, int64_t d, uint64_t rbase, int64_t rbytes,
                                                uint64_t pos, uint64_t line1, int32_t* sE, uint64_t* sD,
                                                int64_t* meta) {
    constexpr int U = 2;
    const int P = p.P;
    const uint64_t* se = p.seg_end + d * P;
    const uint64_t* src = p.seg_src + d * P;
    // twice the segments that a chunk of the row holds on average
    const uint64_t avg = 2 * 16 * (line1 - pos) * (uint64_t)P / (uint64_t)rbytes + 16;
    const int most = avg < kA2avShortWindow ? (int)avg : kA2avShortWindow;
    while (pos < line1) {
        const int64_t o0 = (int64_t)(pos << 4) - (int64_t)rbase;
        const int64_t o = o0 < 0 ? 0 : o0;
        // (few ranks: the whole row, without a search for its first segment)
        const bool whole = P <= kWave;
        const int s0 = whole ? 0 : (int)Group::first_above(se, P, o, &meta[5]);
        const int n = whole ? P : P - s0 < most ? P - s0 : most;
        Group::each([&](int tid) {
            for (int k = tid; k < n; k += kA2avCopyThreads) {
                const int s = s0 + k;
                const int64_t en = (int64_t)se[s], st = s > 0 ? (int64_t)se[s - 1] : 0;
                const int64_t e = en - o;
                sE[k] = (int32_t)(e > INT32_MAX ? INT32_MAX : e < INT32_MIN / 2 ? INT32_MIN / 2 : e);
                sD[k] = src[s] - (rbase + (uint64_t)st);
                if (k == 0) meta[6] = st - o > INT32_MIN / 2 ? st - o : INT32_MIN / 2;
                if (k == n - 1) meta[7] = en;
            }
        });
        const int32_t start0 = (int32_t)Group::uniform(meta[6]);
        const int64_t cover = Group::uniform(meta[7]);
        // lines inside the window's coverage; to the row's end when the window reaches it
        uint64_t pend = s0 + n >= P ? line1 : (rbase + (uint64_t)cover) >> 4;
        if (pend > line1) pend = line1;
        if (pend <= pos) {     // more segments in one line than the window holds
            Group::each([&](int tid) {
                if (tid == 0)
                    a2av_assemble_line(rbase, rbytes, pos, [&](int64_t q) { return a2av_seg_global(p, d, rbase, q); });
            });
            pos++;
            continue;
        }
        const int top = n > 1 ? 1 << (31 - __builtin_clz(n - 1)) : 0;
        auto find = [&](int32_t q) {       // first entry that ends past q
            int k = 0;
            for (int b = top; b > 0; b >>= 1)
                if (k + b <= n - 1 && sE[k + b - 1] <= q) k += b;
            return k;
        };
        Group::each([&](int tid) {
            for (uint64_t base = pos; base < pend; base += (uint64_t)kA2avCopyThreads * U) {
                int32_t q[U];      // window offset of the line's first row byte
                int k[U], kind[U]; // 0 none, 1 one segment, 2 two segments, 3 assemble
                uint32_t cut[U];
                u32x4 v[U], w[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const uint64_t line = base + (uint64_t)u * kA2avCopyThreads + tid;
                    const int64_t off = (int64_t)(line << 4) - (int64_t)rbase;
                    kind[u] = line < pend && off > -16 ? off < 0 || off + 16 > rbytes ? 3 : 1 : 0;
                    q[u] = kind[u] ? (int32_t)(off - o) : 0;
                    if (q[u] < 0) q[u] = 0;
                    k[u] = 0;
                }
                for (int b = top; b > 0; b >>= 1) {
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const int at = k[u] + b <= n - 1 ? k[u] + b : 0;
                        if (at && sE[at - 1] <= q[u]) k[u] = at;
                    }
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    if (kind[u] != 1) continue;
                    const uint64_t la = (base + (uint64_t)u * kA2avCopyThreads + tid) << 4;
                    const int32_t e = sE[k[u]];
                    if (e - q[u] >= 16) {
                        v[u] = gload16(la + sD[k[u]]);
                        continue;
                    }
                    // the next non-empty segment; the one after the line's last byte at most
                    int k2 = k[u] + 1;
                    while (k2 < n - 1 && sE[k2] <= e) k2++;
                    const int32_t st = k[u] > 0 ? sE[k[u] - 1] : start0;
                    if (k2 < n && sE[k2] - e >= 16 && e - st >= 16) {
                        const uint32_t a = (uint32_t)(e - q[u]);       // bytes from the first segment
                        v[u] = gload16(la + a - 16 + sD[k[u]]);
                        w[u] = gload16(la + a + sD[k2]);
                        cut[u] = 16 - a;
                        kind[u] = 2;
                    } else {
                        kind[u] = 3;
                    }
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const uint64_t la = (base + (uint64_t)u * kA2avCopyThreads + tid) << 4;
                    if (kind[u] == 2) v[u] = bytes_from(v[u], w[u], cut[u]);
                    if (kind[u] == 1 || kind[u] == 2) gstore16<NT>(la, v[u]);
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    if (kind[u] != 3) continue;
                    a2av_assemble_line(rbase, rbytes, base + (uint64_t)u * kA2avCopyThreads + tid, [&](int64_t x) {
                        const int j = find((int32_t)(x - o));
                        A2avSegView g;
                        g.st = o + (j > 0 ? sE[j - 1] : start0);
                        g.en = o + sE[j];
                        g.D = sD[j];
                        return g;
                    });
                }
            }
        });
        pos = pend;
    }
}

// FUSE: the first pn.P workgroups plan the next step into pn (a2av_plan_fused); the copy
// workgroups follow them.
template <int U, bool NT, bool DEFER, bool FUSE>
__global__ void __launch_bounds__(kA2avCopyThreads) a2av_copy_kernel(A2avDev p, A2avDev pn) {
    __shared__ int64_t s_st[kA2avWindow];
    __shared__ int64_t s_en[kA2avWindow];
    __shared__ uint64_t s_D[kA2avWindow];
    __shared__ int64_t s_meta[10];
    __shared__ int32_t s_E[DEFER ? 1 : kA2avShortWindow];
    __shared__ uint64_t s_DW[DEFER ? 1 : kA2avShortWindow];
    const int P = p.P;
    const int tid = threadIdx.x;
    const int l = lane();
    uint32_t bid = blockIdx.x, nblk = gridDim.x;
    if constexpr (FUSE) {
        if (bid < (uint32_t)pn.P) {  // block-uniform
            a2av_plan_fused(pn, bid);
            return;
        }
        bid -= (uint32_t)pn.P;
        nblk -= (uint32_t)pn.P;
    }
    uint32_t sb = 0;
    if constexpr (DEFER) {
        sb = (uint32_t)p.straddle_blocks;
        if (bid < sb) {  // block-uniform
            const uint64_t nseg = (uint64_t)P * (uint64_t)P;
            for (uint64_t g = (uint64_t)bid * kA2avCopyThreads + tid; g < nseg;
                 g += (uint64_t)sb * kA2avCopyThreads)
                a2av_straddle_line(p, g);
            return;
        }
    }
    const uint64_t total = p.chunk_off[P];
    const uint64_t C = (uint64_t)p.total_bytes[1];
    // the partial lines at the ends of the long rows: a lane each, in the first blocks
    if constexpr (!DEFER) {
        if (total)
            for (uint64_t g = (uint64_t)bid * kA2avCopyThreads + tid; g < 2 * (uint64_t)P;
                 g += (uint64_t)nblk * kA2avCopyThreads)
                a2av_row_end(p, (int64_t)(g >> 1), (int)(g & 1));
    }
    uint64_t ch = bid - sb;
    for (; ch < total; ch += nblk - sb) {
        // ---- the chunk's row and line range
        if (tid < kWave) {
            const int64_t d = wave_search_le(p.chunk_off, P, ch);
            const uint64_t c = ch - p.chunk_off[d];
            const uint64_t rbase = (uint64_t)(uintptr_t)p.recvbufs[d];
            const uint64_t rbytes = p.row_bytes[d];
            const uint64_t lend = (rbase + rbytes + 15) >> 4;
            // a row's lines start at the 128-byte block holding its first byte, so every
            // wave's 1 KiB slice covers whole 128-byte blocks (lines before the row's first
            // byte write nothing)
            const uint64_t line0 = ((rbase >> 7) << 3) + c * C;
            const uint64_t line1 = line0 + C < lend ? line0 + C : lend;
            if (l == 0) {
                s_meta[0] = d;
                s_meta[1] = (int64_t)rbase;
                s_meta[2] = (int64_t)rbytes;
                s_meta[3] = (int64_t)line0;
                s_meta[4] = (int64_t)line1;
            }
        }
        __syncthreads();
        // block-uniform values read back from LDS: broadcast so that they live in SGPRs
        // (the copy loop is bound by instruction issue; scalar arithmetic is free beside it)
        const int64_t d = bcast(s_meta[0]);
        const uint64_t rbase = (uint64_t)bcast(s_meta[1]);
        const int64_t rbytes = bcast(s_meta[2]);
        const uint64_t line1 = (uint64_t)bcast(s_meta[4]);
        uint64_t pos = (uint64_t)bcast(s_meta[3]);
        while (pos < line1) {
            // ---- window: 64 segments from the one holding the row offset of line `pos`
            if (tid < kWave) {
                int64_t o = (int64_t)(pos << 4) - (int64_t)rbase;
                if (o < 0) o = 0;
                const uint64_t* se = p.seg_end + d * P;
                int64_t s0 = 0;
                if ((int64_t)se[0] <= o) s0 = wave_search_le(se, P, (uint64_t)o) + 1;
                const int64_t s = s0 + l;
                const bool valid = s < P;
                const int64_t en = valid ? (int64_t)se[s] : 0;
                const int64_t st = valid ? (s > 0 ? (int64_t)se[s - 1] : 0) : 0;
                const uint64_t src = valid ? p.seg_src[d * P + s] : 0;
                const bool ne = valid && en > st;
                const uint64_t m = ballot(ne);
                const int k = __popcll(m & (l == 0 ? 0ull : (~0ull >> (64 - l))));
                if (ne) {
                    s_st[k] = st;
                    s_en[k] = en;
                    s_D[k] = src - (rbase + (uint64_t)st);
                }
                const int64_t cover =
                    s0 + kWave >= P ? rbytes : (int64_t)readlane64((uint64_t)en, kWave - 1);
                // the pass takes the lines that end at or before the coverage, at least one
                uint64_t pend = (rbase + (uint64_t)cover) >> 4;
                if (pend > line1) pend = line1;
                int64_t slow = 0;
                if (pend <= pos) {
                    pend = pos + 1;
                    slow = 1;
                }
                // entries that start before the end of the pass's lines bound the searches
                const int64_t pend_off = (int64_t)(pend << 4) - (int64_t)rbase;
                const uint64_t mb = ballot(ne && st < pend_off);
                if (l == 0) {
                    s_meta[5] = __popcll(m);
                    s_meta[6] = (int64_t)pend;
                    s_meta[7] = slow ? 0 : cover;
                    s_meta[8] = slow ? 0 : o;
                    s_meta[9] = __popcll(mb) > 0 ? __popcll(mb) : 1;
                }
            }
            __syncthreads();
            A2avWin w;
            w.st = s_st;
            w.en = s_en;
            w.D = s_D;
            w.cnt = (int)bcast(s_meta[5]);
            w.nsearch = (int)bcast(s_meta[9]);
            const uint64_t pend = (uint64_t)bcast(s_meta[6]);
            w.cover = bcast(s_meta[7]);
            w.lo = bcast(s_meta[8]);
            // each wave copies a contiguous run of 64*U lines, slice by slice, with a
            // wave-uniform cursor over the window (segments only move forward)
            const int wv = tid >> 6;
            for (uint64_t base = pos; base < pend; base += (uint64_t)kA2avCopyThreads * U) {
                const uint64_t wb = base + (uint64_t)wv * kWave * U;
                if (wb >= pend) continue;
                int64_t off0 = (int64_t)(wb << 4) - (int64_t)rbase;
                int kc = bcast(a2av_seg_lds(s_st, w.nsearch, off0 > w.lo ? off0 : w.lo));
                // entries kc and kc + 1 (ends and source offsets), cached in SGPRs
                int kc1 = kc + 1 < w.cnt ? kc + 1 : kc;
                int64_t Ekc = bcast(s_en[kc]), Ekc1 = bcast(s_en[kc1]);
                uint64_t Dkc = bcast(s_D[kc]), Dkc1 = bcast(s_D[kc1]);
                u32x4 v[U];
                int kind[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const uint64_t sl = wb + (uint64_t)u * kWave;  // slice's first line
                    const uint64_t line = sl + l;
                    kind[u] = line < pend ? 2 : 0;
                    if (sl >= pend) continue;  // wave-uniform
                    const int64_t soff = (int64_t)(sl << 4) - (int64_t)rbase;
                    // move the cursor to the entry holding the slice's first byte: a few
                    // steps forward, or a search when the slice starts further ahead
                    if (soff >= Ekc && kc + 1 < w.nsearch) {
                        if (kc + 3 < w.nsearch && soff >= bcast(s_en[kc + 3]))
                            kc = bcast(a2av_seg_lds(s_st, w.nsearch, soff));
                        else
                            while (kc + 1 < w.nsearch && soff >= bcast(s_en[kc])) kc++;
                        kc1 = kc + 1 < w.cnt ? kc + 1 : kc;
                        Ekc = bcast(s_en[kc]);
                        Dkc = bcast(s_D[kc]);
                        Ekc1 = bcast(s_en[kc1]);
                        Dkc1 = bcast(s_D[kc1]);
                    }
                    const int64_t off = soff + 16 * l;
                    if (soff + 16 * kWave <= Ekc) {
                        // the whole slice lies in entry kc (the common case): one uniform
                        // source offset, no per-lane selection, no LDS access
                        if (line < pend && off >= w.lo) {
                            v[u] = gload16((line << 4) + Dkc);
                            kind[u] = 1;
                        }
                        continue;
                    }
                    if (!DEFER && soff + 16 * kWave <= Ekc1) {
                        // the slice spans entries kc and kc + 1: a lane's line lies in one of
                        // them or straddles their boundary (one lane at most)
                        if (line < pend && off >= w.lo) {
                            const uint64_t la = line << 4;
                            if (off + 16 <= Ekc || off >= Ekc) {
                                v[u] = gload16(la + (off < Ekc ? Dkc : Dkc1));
                                kind[u] = 1;
                            } else if constexpr (!DEFER) {
                                if (((Ekc - off) & 3) == 0 && ((la + Dkc) & 3) == 0 && ((la + Dkc1) & 3) == 0) {
                                    v[u] = u32x4{
                                        *(const GPUMPI_GLOBAL uint32_t*)(uintptr_t)(la + (off < Ekc ? Dkc : Dkc1)),
                                        *(const GPUMPI_GLOBAL uint32_t*)(uintptr_t)(la + 4 + (off + 4 < Ekc ? Dkc : Dkc1)),
                                        *(const GPUMPI_GLOBAL uint32_t*)(uintptr_t)(la + 8 + (off + 8 < Ekc ? Dkc : Dkc1)),
                                        *(const GPUMPI_GLOBAL uint32_t*)(uintptr_t)(la + 12 + (off + 12 < Ekc ? Dkc : Dkc1))};
                                    kind[u] = 1;
                                }
                            }
                        }
                        continue;
                    }
                    if (!(line < pend && off >= w.lo && off + 16 <= w.cover)) continue;
                    // this lane's entry: the cursor or one of the next three, else a search
                    int kb = kc;
                    if (kc + 3 < w.cnt && off >= s_en[kc + 3]) kb = a2av_seg_lds(s_st, w.nsearch, off);
                    const int k1 = kb + 1 < w.cnt ? kb + 1 : kb, k2 = kb + 2 < w.cnt ? kb + 2 : k1,
                              k3 = kb + 3 < w.cnt ? kb + 3 : k2;
                    const int64_t e0 = s_en[kb], e1 = s_en[k1], e2 = s_en[k2], e3 = s_en[k3];
                    const uint64_t D0 = s_D[kb], D1 = s_D[k1], D2 = s_D[k2], D3 = s_D[k3];
                    const uint64_t la = line << 4;
                    const int j = (off >= e0) + (off >= e1) + (off >= e2);
                    const int64_t ej = j == 0 ? e0 : j == 1 ? e1 : j == 2 ? e2 : e3;
                    const uint64_t Dj = j == 0 ? D0 : j == 1 ? D1 : j == 2 ? D2 : D3;
                    if (off + 16 <= ej) {
                        v[u] = gload16(la + Dj);
                        kind[u] = 1;
                        continue;
                    }
                    if constexpr (DEFER) continue;
                    // the line straddles segments: one dword from the segment holding it
                    uint64_t a[4];
                    bool ok = true;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int64_t q = off + 4 * i;
                        const int ji = (q >= e0) + (q >= e1) + (q >= e2);
                        const int64_t eq = ji == 0 ? e0 : ji == 1 ? e1 : ji == 2 ? e2 : e3;
                        const uint64_t Dq = ji == 0 ? D0 : ji == 1 ? D1 : ji == 2 ? D2 : D3;
                        a[i] = la + 4 * i + Dq;
                        ok = ok && (a[i] & 3) == 0 && q + 4 <= eq;
                    }
                    if (ok) {
                        v[u] = u32x4{*(const GPUMPI_GLOBAL uint32_t*)(uintptr_t)a[0],
                                     *(const GPUMPI_GLOBAL uint32_t*)(uintptr_t)a[1],
                                     *(const GPUMPI_GLOBAL uint32_t*)(uintptr_t)a[2],
                                     *(const GPUMPI_GLOBAL uint32_t*)(uintptr_t)a[3]};
                        kind[u] = 1;
                    }
                }
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (kind[u] == 1) gstore16<NT>((wb + (uint64_t)u * kWave + l) << 4, v[u]);
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (kind[u] == 2)
                        a2av_boundary_line<DEFER>(p, d, rbase, rbytes, w, wb + (uint64_t)u * kWave + l);
            }
            __syncthreads();
            pos = pend;
        }
    }
    // the short rows' chunks follow the long rows' in a loop of their own: in one loop, the
    // registers of the loads above stay live through this path (115 instead of 87)
    if constexpr (!DEFER) {
        const uint64_t shorts = p.short_off[P], S = (uint64_t)p.total_bytes[2];
        for (; ch - total < shorts; ch += nblk) {
            if (tid < kWave) {
                if (P <= kWave) {
                    // every row's words in one round of loads
                    const int r = l < P ? l : P - 1;
                    const uint64_t off = p.short_off[r], base = (uint64_t)(uintptr_t)p.recvbufs[r], word = p.row_bytes[r];
                    const int d = 63 - __builtin_clzll(ballot(l < P && off <= ch - total));
                    if (l == d) {
                        s_meta[0] = d;
                        s_meta[1] = (int64_t)(ch - total - off);
                        s_meta[2] = (int64_t)base;
                        s_meta[3] = (int64_t)word;
                    }
                } else {
                    const int64_t d = wave_search_le(p.short_off, P, ch - total);
                    if (l == 0) {
                        s_meta[0] = d;
                        s_meta[1] = (int64_t)(ch - total - p.short_off[d]);
                        s_meta[2] = (int64_t)(uintptr_t)p.recvbufs[d];
                        s_meta[3] = (int64_t)p.row_bytes[d];
                    }
                }
            }
            __syncthreads();
            const int64_t d = bcast(s_meta[0]);
            const uint64_t c = (uint64_t)bcast(s_meta[1]);
            const uint64_t rbase = (uint64_t)bcast(s_meta[2]);
            const int64_t rbytes = (int64_t)((uint64_t)bcast(s_meta[3]) & ~kA2avShortRow);
            const uint64_t lend = (rbase + (uint64_t)rbytes + 15) >> 4;
            const uint64_t line0 = ((rbase >> 7) << 3) + c * S;
            const uint64_t line1 = line0 + S < lend ? line0 + S : lend;
            a2av_copy_short<NT, A2avGroup>(p, d, rbase, rbytes, line0, line1, s_E, s_DW, s_meta);
        }
    }
}

}  // namespace gpumpi
