// The bucket plan with the tiling that it takes where memory for the table of counts is not to be
// had (one workgroup per rank, several tiles in turn), and with two tiles per workgroup, against
// a stable bucketing on the host: every scatter kernel's loop over tiles.
#include "runtime/bucket_plan.h"

#include <cstdio>
#include <random>
#include <vector>

using namespace gpumpi;

static int run(int P, int64_t n, int key_bits, int bucket_bits, int turns) {
    const int nb = 1 << bucket_bits, shift = key_bits - bucket_bits;
    std::printf("P %d n %lld bits %d/%d turns %d\n", P, (long long)n, key_bits, bucket_bits, turns);
    std::fflush(stdout);
    BucketTiling t = bucket_tiling(P, n, nb, turns == 0);
    if (turns) {
        const uint32_t all = (uint32_t)((n + t.base - 1) / t.base);
        t.subs = (uint32_t)turns;
        t.tiles = (all + t.subs - 1) / t.subs;
    }
    const size_t N = (size_t)P * (size_t)n;
    std::vector<uint32_t> keys(N), want(N), got(N);
    std::mt19937 rng((unsigned)(P + n));
    for (uint32_t& k : keys) k = rng() >> (32 - key_bits) & (rng() & 3 ? ~0u : 0xFFu);
    std::vector<int32_t> wc((size_t)P * P), wd((size_t)P * P), gc((size_t)P * P), gd((size_t)P * P), lo(P), hi(P);
    std::vector<std::vector<uint32_t>> pre(P, std::vector<uint32_t>((size_t)nb + 1, 0));
    for (int r = 0; r < P; r++) {
        for (int64_t i = 0; i < n; i++) pre[r][(keys[r * n + i] >> shift) + 1]++;
        for (int b = 0; b < nb; b++) pre[r][b + 1] += pre[r][b];
        std::vector<uint32_t> at(pre[r]);
        for (int64_t i = 0; i < n; i++) want[r * n + at[keys[r * n + i] >> shift]++] = keys[r * n + i];
    }
    uint32_t *dk, *dout;
    int32_t* dx;
    void* scratch;
    const size_t xs = 2 * (size_t)P * P + 2 * P;
    if (hipMalloc((void**)&dk, 4 * N) != hipSuccess || hipMalloc((void**)&dout, 4 * N) != hipSuccess ||
        hipMalloc((void**)&dx, 4 * xs) != hipSuccess || hipMalloc(&scratch, bucket_scratch_bytes(t, P, nb)) != hipSuccess ||
        hipMemcpy(dk, keys.data(), 4 * N, hipMemcpyHostToDevice) != hipSuccess)
        return 1;
    bucket_plan_launch(t, dk, P, n, shift, nb, scratch, dout, dx, dx + (size_t)P * P, dx + 2 * (size_t)P * P,
                       dx + 2 * (size_t)P * P + P, 0);
    std::vector<int32_t> x(xs);
    if (hipGetLastError() != hipSuccess || hipMemcpy(got.data(), dout, 4 * N, hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(x.data(), dx, 4 * xs, hipMemcpyDeviceToHost) != hipSuccess)
        return 1;
    hipFree(dk);
    hipFree(dout);
    hipFree(dx);
    hipFree(scratch);
    int bad = got != want;
    const int32_t *l = &x[2 * (size_t)P * P], *h = l + P;
    for (int r = 0; r < P; r++)
        for (int d = 0; d < P; d++) {
            const bool some = l[d] <= h[d];
            const int32_t c = some ? (int32_t)(pre[r][h[d] + 1] - pre[r][l[d]]) : 0;
            const int32_t at = (int32_t)(some ? pre[r][l[d]] : pre[r][nb]);
            bad |= x[(size_t)r * P + d] != c || x[(size_t)P * P + (size_t)r * P + d] != at;
        }
    if (bad) std::printf("wrong\n");
    return bad;
}

int main() {
    int bad = 0;
    // 16 and 4 keys per thread of 1024 threads, of 512 (more than 1024 buckets)
    for (int turns : {0, 2}) {
        bad |= run(520, 16385, 20, 10, turns);
        bad |= run(3, 20001, 18, 9, turns);
        bad |= run(1, 4097, 11, 9, turns);
        bad |= run(70, 66000, 20, 12, turns);
        bad |= run(5, 10001, 20, 11, turns);
        bad |= run(2, 2048, 13, 12, turns);
        if (bad) break;
    }
    if (!bad) std::printf("all equal\n");
    return bad;
}
