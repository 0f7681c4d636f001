// z2h_rules.h — host-side choices between two shapes of one matmul kernel, as plain functions of sizes (both sides
// give the same bits, so the lines are about speed alone).
#pragma once
#include <cmath>
#include <cstdint>

namespace z2r {

// F16 expert matmuls of wide launches: token tiles of 128 rows instead of 64. Both keep two blocks on a compute unit, so
// a launch takes whole rounds of 2 n_cu blocks. Tall tiles read the weights half as often but a round of them costs
// more: relative to the first round of 64-row tiles, each further one 0.53, the first of 128 rows 1.28, each further
// one 0.78 (32 experts of 2048 x 1536, gate/up: 90 + 48 us per round against 115 + 70; down 63 + 45 against 80 + 70).
// So tall tiles pay where they save rounds, and lose where the launch does not fill the chip (4 experts, 512
// routes each: 46 us against 68). A launch of `items` routes over E experts has about items / G + E / 2 tiles of G
// rows; the experts' loads are not known here, so the counts are taken 6% low and 4% high, and below 112 routes per
// expert uneven loads leave the estimate too far off (Zipf 1.2, 75 routes: 130 us against 147). On 15 shapes of 4 to
// 128 experts, even and Zipf loads, 32 to 1000 routes per expert, the rule's choice of tall tiles gained 15% on average
// and lost nowhere.
//   row_blocks: blocks along the output rows
inline bool f16_tall_tiles(int64_t row_blocks, int64_t items, int E, int n_cu) {
    if (items < 112ll * E) return false;
    const double w = (double) row_blocks / (2.0 * n_cu);
    const double n64 = std::ceil(0.94 * w * ((double) items / 64 + 0.5 * E)), n128 = std::ceil(1.04 * w * ((double) items / 128 + 0.5 * E));
    return 1.28 + 0.78 * (n128 - 1) < 1.0 + 0.53 * (n64 - 1);
}

} // namespace z2r
