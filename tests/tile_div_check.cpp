// tile_div_rcp (ee_tile_div.h) against integer division, with the reciprocal at -1, 0 and +1 ulp:
//   every t < 2^23 with every multiple of t up to 2^23 and its two neighbours;
//   up to 2^30, t near powers of two and pseudo-random ones, at multiples of t, their neighbours
//   and pseudo-random i.
// Exit status 0 iff no quotient differs.  Built and run by tests/test_tile_div_exhaustive.py.
#include <cmath>
#include <cstdint>
#include <cstdio>

#include "common/ee_tile_div.h"

static int64_t check(int64_t i, int t, int64_t top) {
    static thread_local int shown = 0;
    if (i < 0 || i >= top) return 0;
    int64_t bad = 0;
    const float r = 1.0f / (float)t;
    const float rs[3] = {nextafterf(r, 0.0f), r, nextafterf(r, 2.0f)};
    for (float rt : rs) {
        const int q = tile_div_rcp((int)i, t, rt);
        if (q != (int)(i / t)) {
            ++bad;
            if (shown++ < 5) std::printf("mismatch i %lld t %d: %d, not %lld\n", (long long)i, t, q, (long long)(i / t));
        }
    }
    return bad;
}

int main() {
    const int64_t top = int64_t(1) << 23, big = int64_t(1) << 30;
    int64_t bad = 0, n = 0;
#pragma omp parallel for schedule(dynamic, 256) reduction(+ : bad, n)
    for (int t = 1; t < (int)top; ++t) {
        for (int64_t i = 0; i <= top; i += t)
            for (int d = -1; d <= 1; ++d, ++n) bad += check(i + d, t, top);
    }
#pragma omp parallel for schedule(dynamic, 64) reduction(+ : bad, n)
    for (int k = 0; k < 40000; ++k) {
        uint64_t x = 0x9e3779b97f4a7c15ull * (uint64_t)(k + 1);
        auto next = [&] { x ^= x << 13; x ^= x >> 7; x ^= x << 17; return x; };
        const int e = k % 30;
        int64_t t = k < 3000 ? (int64_t(1) << e) + k / 30 - 50 : int64_t(next() >> 34 >> (k % 29));
        if (t < 1 || t >= big) continue;
        for (int j = 0; j < 300; ++j) {
            const int64_t i = int64_t(next() >> 34), m = i / t * t;
            bad += check(i, (int)t, big);
            for (int d = -1; d <= 1; ++d) bad += check(m + d, (int)t, big);
            n += 4;
        }
        for (int d = 1; d < 4; ++d, ++n) bad += check(big - d, (int)t, big);
    }
    std::printf("quotients %lld mismatches %lld\n", (long long)n, (long long)bad);
    return bad ? 1 : 0;
}
