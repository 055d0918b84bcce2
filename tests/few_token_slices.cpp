// The few-token prefill kernel's slices (few_token_slices.h) for every row length around the limit and a
// spread of the others, row counts and chip sizes: each slice has 1 to kSkMaxSteps steps, they cover the
// row, the workspace covers them, and their count fits the arrival counter.
#include <cstdio>
#include <initializer_list>

#include "few_token_slices.h"

using namespace tqhip;

int main() {
    int bad = 0, longest = 0;
    const auto check = [&](int M, int K, int cus) {
        if (!skinny_row_fits(K)) return;
        longest = std::max(longest, K);
        const SkinnyGeom g = skinny_geom(M, K, cus);
        // the counter after KS - 1 arrivals, as the last one reads it, must say KS - 1
        const unsigned long long count = static_cast<unsigned long long>(g.KS - 1) << kArrivalShift >> kArrivalShift;
        const unsigned long long full = static_cast<unsigned long long>(g.KS) << kArrivalShift >> kArrivalShift;
        bool ok = count == static_cast<unsigned long long>(g.KS - 1) && full == static_cast<unsigned long long>(g.KS);
        ok = ok && g.KS >= 1 && g.KS <= g.T && g.smax >= 1 && g.smax <= kSkMaxSteps && g.part_bytes <= g.room;
        for (int ks = 0; ok && ks < g.KS; ++ks) {
            const int ns = static_cast<int>((ks + 1LL) * g.T / g.KS - 1LL * ks * g.T / g.KS);
            ok = ns >= 1 && ns <= g.smax && (ks + 1) * g.T / g.KS == (ks + 1LL) * g.T / g.KS;  // (the kernel's int arithmetic)
        }
        if (!ok && bad++ < 10) std::printf("M %d K %d CUs %d: %d slices of %d steps\n", M, K, cus, g.KS, g.T);
    };
    for (int cus : {1, 64, 256, 304})
        for (int M : {1, 128, 129, 896, 4096, 70000, 151936}) {
            for (int K = 4; K <= 32768; K += 60) check(M, K, cus);
            for (int K = 113000; K <= 116000; K += 4) check(M, K, cus);
            for (int K = 40000; K < 29000000; K += K / 7 / 4 * 4) check(M, K, cus);
        }
    if (bad == 0 && longest >= kMaxSlices * kSkMaxSteps * 64 - 64) std::printf("ok slices, rows up to %d\n", longest);
    return bad != 0;
}
