// Compares the 64-bit forms of the systematic draws (component_key,
// SysThresholds of pf_common.hpp) with their 128-bit definitions, at the ends
// of their ranges and at random inside them.  Host only; prints the number of
// comparisons and exits 1 at the first difference.
#include <cinttypes>
#include <cstdio>
#include <random>

#include "../../mkfbodytracker_pdaf_amd/csrc/pf_common.hpp"

using namespace mkfbt;

int main()
{
    std::mt19937_64 rng(2024);
    long long n = 0;
    auto between = [&](uint64_t lo, uint64_t hi) { return lo + rng() % (hi - lo + 1); };
    auto log_size = [&](int bits) { return between(1, (uint64_t)1 << between(0, bits)); };
    const uint32_t edges[] = {0u, 1u, 0x7fffffffu, 0x80000000u, 0xffffffffu};
    for (int trial = 0; trial < 20000; ++trial) {
        // outputs: f_i = floor((i 2^32 + U) total / (N 2^32))
        const uint64_t N = trial % 4 == 0 ? (trial % 8 ? (uint64_t)1 << 26 : 1) : log_size(26);
        const uint64_t total = trial % 5 == 0 ? (uint64_t)1 << 52 : log_size(52);
        const uint32_t U = trial % 3 == 0 ? edges[trial % 5] : (uint32_t)rng();
        const SysThresholds f(total, U, (uint32_t)N);
        for (int r = 0; r < 12; ++r) {
            const uint64_t i = r == 0 ? 0 : (r == 1 ? N - 1 : rng() % N);
            const u128 t = (((u128)i << 32) | U) * total;
            if ((u128)f((uint32_t)i) != t / ((u128)N << 32)) {
                printf("threshold: N=%" PRIu64 " total=%" PRIu64 " U=%u i=%" PRIu64 "\n", N, total, U, i);
                return 1;
            }
            ++n;
        }
        // components: C N 2^32 <= (j 2^32 + U) T exactly when key <= j 2^32 + U
        const uint64_t T = between(1, (uint64_t)1 << 40), C = trial % 7 == 0 ? T : rng() % (T + 1);
        const uint64_t M = log_size(20), key = component_key(C, T, M);
        for (int r = 0; r < 12; ++r) {
            const uint64_t at = r < 3 ? key + r - 1 : (rng() % M) << 32 | U;
            const uint64_t j = at >> 32;
            if (key == 0 && r == 0) continue;
            const bool want = (u128)C * ((u128)M << 32) <= (u128)at * T;
            if ((key <= at) != want) {
                printf("component: M=%" PRIu64 " T=%" PRIu64 " C=%" PRIu64 " j=%" PRIu64 "\n", M, T, C, j);
                return 1;
            }
            ++n;
        }
    }
    printf("%lld comparisons\n", n);
    return 0;
}
