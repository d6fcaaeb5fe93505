// Every quotient A / D of 24-bit significands that lies within |r| <= 8 steps of a
// midpoint of two adjacent floats, through hs_div_fast (hs_div.h) and the host's
// IEEE division.  A step is 1 / (2^s D), s = 24 for A >= D and 25 below: the
// quotients are the solutions of  2^s A = M D + r  with M odd in [2^24, 2^25),
// found for each D from the inverse of its odd part modulo 2^s.  Prints the
// counts; exit status 1 on a mismatch or a refused quotient.
#include <cmath>
#include <cstdint>
#include <cstdio>

#include "../hindemith_amd/csrc/hs_div.h"

int main() {
    long long n = 0, bad = 0;
    const uint64_t lo = 1ull << 23, hi = 1ull << 24;
    for (uint64_t D = lo; D < hi; ++D) {
        const int t = __builtin_ctzll(D);
        const uint32_t odd = (uint32_t)(D >> t);
        uint32_t inv = odd;
        for (int i = 0; i < 5; ++i) inv *= 2u - odd * inv;
        const float d = (float)D, y = hmx::hs_recip(d * 0x1p-23f);
        for (int s = 24; s <= 25; ++s)
            for (int r = -8; r <= 8; ++r) {
                if (r == 0 || t > 3 || r % (1 << t)) continue;  // D's factor 2^t divides r
                const uint64_t step = 1ull << (s - t);
                // M odd' = -r / 2^t (mod 2^(s - t))
                const uint64_t m0 = ((uint64_t)(uint32_t)(-(r / (1 << t))) * inv) & (step - 1);
                if (!(m0 & 1)) continue;
                for (uint64_t M = m0; M < (1ull << 25); M += step) {
                    if (M < (1ull << 24)) continue;
                    const int64_t num = (int64_t)(M * D) + r;
                    if (num & ((1ll << s) - 1)) continue;
                    const uint64_t A = (uint64_t)(num >> s);
                    if (A < lo || A >= hi || (s == 24) != (A >= D)) continue;
                    const float a = (float)A * 0x1p-23f, b = d * 0x1p-23f;
                    float q;
                    ++n;
                    if (!hmx::hs_div_fast(a, b, y, q) || q != a / b) ++bad;
                }
            }
    }
    std::printf("quotients %lld mismatches %lld\n", n, bad);
    return bad == 0 && n > 40000000 ? 0 : 1;
}
