// few_token_slices.h -- how the few-token prefill kernel (i4_matmul.hip, section 3) cuts K into slices, and the
// limit that its arrival counters put on them. No device code: compiled with g++ by the CPU tests.
#pragma once

#include <algorithm>
#include <cstddef>

namespace tqhip {

// A tile's arrival counter (64 bits, zero between launches): bits kArrivalShift.. count the slices that
// have stored their partial; bits 4 p .. 4 p + 3 hold 1 + the XCD of slice p's writer, p < kXccSlots.
constexpr int kArrivalShift = 56;
constexpr int kXccSlots = kArrivalShift / 4;
constexpr int kMaxSlices = (1 << (64 - kArrivalShift)) - 1;  // the count of the last arrival but one fits

constexpr int kSkRows = 128;           // rows of a tile
constexpr int kSkTile = kSkRows * 32;  // floats of one partial
constexpr int kSkMaxSteps = 7;         // 64-element steps of a slice: a row's (9 dwords a step) within one 64-lane DMA

struct SkinnyGeom {
    int tiles, T, KS, smax;
    size_t part_bytes;  // the partial products
    size_t room;        // the partials of as many slices as may be taken: what a fixed workspace must hold
};

// At most about 1.9 workgroups per CU (all resident at once), kSkMaxSteps steps per slice and one
// slice per step; among these the slices with the least estimated time: the tile's last
// workgroup reads its KS partials of 16 KB alone, 0.33 us each, a step of a slice takes 0.28 us
// (fitted on MI355X to 896x4864 with 70 / 37 / 22 / 11 slices: 30.0, 19.5, 14.6, 11.7 us). Filling the
// chip instead, us -> this rule, 8 tokens: 896x896 10.1 -> 7.7, 4864x896 12.0 -> 8.3, 896x4864
// 30.2 -> 11.7, 2560x4096 19.6 -> 12.0, 2048x2048 17.9 -> 9.4; 9728x2560 and 151936x896 the same. Over 14 shapes
// from 128x896 to 18944x3584 at 2, 8 and 32 tokens one is slower, 2560x9728 at 32: 23.4 -> 23.7.
inline SkinnyGeom skinny_geom(int M, int K, int cus) {
    SkinnyGeom g;
    g.tiles = (M + kSkRows - 1) / kSkRows;
    g.T = (K + 63) / 64;
    const int ks = std::max((19 * cus + 5 * g.tiles) / (10 * g.tiles), (g.T + kSkMaxSteps - 1) / kSkMaxSteps);
    const int most = std::max(1, std::min({ks, g.T, kMaxSlices}));
    g.KS = most;
    float best = 0.f;
    for (int k = most; k >= 1 && (g.T + k - 1) / k <= kSkMaxSteps; --k) {
        const long rounds = (static_cast<long>(g.tiles) * k + 2 * cus - 1) / (2 * cus);
        const float cost = (k > 1 ? 0.33f * k : 0.f) + 0.28f * ((g.T + k - 1) / k) * rounds;
        if (k == most || cost < best) {
            best = cost;
            g.KS = k;
        }
    }
    g.smax = (g.T + g.KS - 1) / g.KS;
    g.room = static_cast<size_t>(g.tiles) * most * kSkTile * sizeof(float);
    g.part_bytes = static_cast<size_t>(g.tiles) * g.KS * kSkTile * sizeof(float);
    return g;
}

// Rows that so many slices cover (114240 elements): a longer one takes the tiled GEMM, whose steps are not
// limited. With more slices the count would wrap, no workgroup would be the last, and Y would stay
// unwritten and the counters non-zero.
inline bool skinny_row_fits(int K) { return K > 0 && (K - 1) / 64 + 1 <= kMaxSlices * kSkMaxSteps; }

}  // namespace tqhip
