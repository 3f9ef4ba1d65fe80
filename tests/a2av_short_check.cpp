// The short rows' copy, its line assembly and the long rows' ends (runtime/batched.h) on the CPU: the
// code of the kernels, its threads one after the other, over random layouts.  Every byte of every
// row must come out as the plain exchange gives it and nothing beside the rows may be written;
// the sanitizers stop on a load outside its segment.
#include "runtime/batched.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <random>
#include <vector>

using namespace gpumpi;

struct Serial {
    template <class F>
    static void each(F f) {
        for (int tid = 0; tid < kA2avCopyThreads; tid++) f(tid);
    }
    static int32_t uniform(int32_t v) { return v; }
    static int64_t uniform(int64_t v) { return v; }
    static int64_t first_above(const uint64_t* se, int64_t n, int64_t o, int64_t* slot) {
        int64_t k = 0;
        while (k < n && (int64_t)se[k] <= o) k++;
        return *slot = k;
    }
};

// One row of P segments of the given sizes, its receive buffer at `phase` past a 128-byte block.
// Short: copied in chunks of `lines` lines.  Otherwise only its two ends, as a long row.
static int run(const std::vector<uint64_t>& size, uint64_t phase, uint64_t lines, bool is_short, unsigned seed) {
    const int P = (int)size.size();
    std::mt19937 rng(seed);
    std::vector<uint64_t> end(P), src(P);
    std::vector<std::unique_ptr<unsigned char[]>> seg(P);
    uint64_t bytes = 0;
    for (int s = 0; s < P; s++) {
        const uint64_t shift = rng() & 1 ? rng() % 16 : 0;     // sources at any alignment
        seg[s].reset(new unsigned char[size[s] + shift]);      // ends with its last byte
        for (uint64_t i = 0; i < size[s]; i++) seg[s][shift + i] = (unsigned char)rng();
        src[s] = (uint64_t)(uintptr_t)(seg[s].get() + shift);
        bytes += size[s];
        end[s] = bytes;
    }
    if (bytes == 0) return 0;
    const uint64_t room = (phase + bytes + 127) / 128 * 128 + 256;
    unsigned char* area = (unsigned char*)std::aligned_alloc(128, room);
    std::memset(area, 0xA5, room);
    unsigned char* recv = area + 128 + phase;
    std::vector<unsigned char> want(area, area + room);
    for (int s = 0; s < P; s++)
        if (size[s]) std::memcpy(&want[128 + phase + end[s] - size[s]], (const void*)(uintptr_t)src[s], size[s]);
    A2avDev p{};
    uint64_t word = is_short ? bytes | kA2avShortRow : bytes;
    char* rb[1] = {(char*)recv};
    p.P = P;
    p.elem = 1;
    p.seg_end = end.data();
    p.seg_src = src.data();
    p.row_bytes = &word;
    p.recvbufs = rb;
    const uint64_t rbase = (uint64_t)(uintptr_t)recv, lend = (rbase + bytes + 15) >> 4;
    if (is_short) {
        std::unique_ptr<int32_t[]> sE(new int32_t[kA2avShortWindow]);
        std::unique_ptr<uint64_t[]> sD(new uint64_t[kA2avShortWindow]);
        std::unique_ptr<int64_t[]> meta(new int64_t[10]);
        for (uint64_t l0 = (rbase >> 7) << 3; l0 < lend; l0 += lines)
            a2av_copy_short<false, Serial>(p, 0, rbase, (int64_t)bytes, l0, l0 + lines < lend ? l0 + lines : lend, sE.get(),
                                           sD.get(), meta.get());
    } else {
        a2av_row_end(p, 0, 0);
        a2av_row_end(p, 0, 1);
        // the lines inside are the copy loop's
        for (uint64_t i = 0; i < bytes; i++) {
            const uint64_t line = (rbase + i) >> 4;
            if (line << 4 >= rbase && (line << 4) + 16 <= rbase + bytes) {
                if (recv[i] != 0xA5) return 1;
                recv[i] = want[128 + phase + i];
            }
        }
    }
    const int bad = std::memcmp(area, want.data(), room) != 0;
    std::free(area);
    return bad;
}

int main() {
    // every cut of two 16-byte vectors, every short load
    unsigned char v[32];
    for (int i = 0; i < 32; i++) v[i] = (unsigned char)(17 * i + 3);
    u32x4 a, b;
    std::memcpy(&a, v, 16);
    std::memcpy(&b, v + 16, 16);
    for (uint32_t at = 0; at <= 16; at++) {
        const u32x4 x = bytes_from(a, b, at);
        if (std::memcmp(&x, v + at, 16)) return std::printf("bytes_from at %u\n", at), 1;
    }
    for (uint32_t n = 0; n < 16; n++) {
        std::unique_ptr<unsigned char[]> exact(new unsigned char[n + 1]);
        std::memcpy(exact.get() + 1, v, n);
        const u32x4 x = load_bytes((uint64_t)(uintptr_t)(exact.get() + 1), n);
        unsigned char y[16] = {};
        std::memcpy(y, v, n);
        if (std::memcmp(&x, y, 16)) return std::printf("load_bytes %u\n", n), 1;
    }
    std::mt19937 rng(11);
    struct Kind { int P; double mean, empty; };
    // up to 64 ranks the window is the whole row; more ranks search; more than a window holds
    const Kind kinds[] = {{1, 5, 0}, {2, 4, 0}, {2, 14, 0}, {1, 70000, 0}, {3, 700, 0.3}, {16, 40, 0.3}, {40, 17, 0.3}, {64, 1, 0.3}, {64, 900, 0.1}, {64, 30000, 0.2},
                          {65, 30, 0.3}, {200, 157, 0.1}, {200, 3000, 0.1}, {700, 3, 0.3}, {700, 300, 0.7}, {1300, 2, 0.3}, {2000, 40, 0.0}};
    for (const Kind& k : kinds)
        for (unsigned seed = 0; seed < 6; seed++) {
            auto phase = [&] { return seed % 3 ? rng() % 128 : rng() % 8 * 16; };
            std::poisson_distribution<int> d(k.mean);
            std::vector<uint64_t> size(k.P);
            for (uint64_t& x : size) x = (rng() % 1000) / 1000.0 < k.empty ? 0 : (uint64_t)d(rng);
            if (k.P > 600 && seed % 2)
                for (int s = 20; s < 20 + kA2avShortWindow + 30; s++) size[s] = 0;     // more empty ones in a line than a window holds
            if (seed == 3) size[k.P / 2] += 100000;      // one long among the short
            for (uint64_t lines : {kA2avShortLines, kA2avShortMost, (uint64_t)64})
                if (run(size, phase(), lines, true, seed))
                    return std::printf("short row: P %d mean %g seed %u lines %u\n", k.P, k.mean, seed, (unsigned)lines), 1;
            if (run(size, phase(), 0, false, seed))
                return std::printf("row ends: P %d mean %g seed %u\n", k.P, k.mean, seed), 1;
        }
    return 0;
}
