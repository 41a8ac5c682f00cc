// The three-operation division of the final passes, q = a inv, q + (a - q s) inv with
// inv = 1 / s correctly rounded, against the IEEE quotient, where it could go wrong: on
// every pair of significands a, s in [2^23, 2^24) whose quotient lies within
// 16 / (2 s) units in the last place of a midpoint Q + 1/2 (the corrected value is off by
// at most 4 * 2^-25 units before it is rounded, a quarter of that).
//
// Those are the solutions of a 2^S - (2 Q + 1) s = N with 0 < |N| <= 16, S = 24 for
// a >= s and 25 below: with s = o 2^t (o odd), N has to be a multiple of 2^t, and
// 2 Q + 1 is -(N / 2^t) / o modulo 2^(S - t).  N = 0 has no solution (a midpoint would
// need 25 significant bits from 24).
//
// Prints the pairs, the wrong quotients, and the wrong ones without the correction.
#include <cmath>
#include <cstdint>
#include <cstdio>

int main() {
    long long pairs = 0, wrong = 0, plain = 0;
#pragma omp parallel for schedule(dynamic, 4096) reduction(+ : pairs, wrong, plain)
    for (uint32_t si = 1u << 23; si < 1u << 24; ++si) {
        const float s = (float)si, inv = 1.f / s;
        const int t = __builtin_ctz(si);
        const uint64_t o = si >> t;
        uint64_t oi = o;  // 1 / o modulo 2^64, by Newton
        for (int k = 0; k < 6; ++k) oi *= 2u - o * oi;
        for (int S = 24; S <= 25; ++S) {
            const int m = S - t;
            if (m < 1) continue;
            const uint64_t mod = 1ull << m;
            for (int N = -16; N <= 16; ++N) {
                if (N == 0 || (N & ((1 << t) - 1))) continue;
                const int64_t n = N / (1 << t);
                for (uint64_t z = (uint64_t)(-n) * oi & (mod - 1); z < 1ull << 25; z += mod) {
                    if (!(z & 1u) || z < 1ull << 24) continue;  // 2 Q + 1, Q of 24 bits
                    const uint64_t ai = (z * o + (uint64_t)n) >> m;
                    if (ai < 1u << 23 || ai >= 1u << 24) continue;
                    const float a = (float)ai, q0 = a * inv, q = std::fmaf(std::fmaf(-q0, s, a), inv, q0);
                    ++pairs;
                    wrong += q != a / s;
                    plain += q0 != a / s;
                }
            }
        }
    }
    std::printf("%lld %lld %lld\n", pairs, wrong, plain);
    return 0;
}
