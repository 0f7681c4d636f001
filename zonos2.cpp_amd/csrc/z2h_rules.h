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

// Dense F16 matmuls of at most 64 token rows: k_gemm_f16_few (16 or 32 weight rows per block, the whole K range requested at
// once) instead of k_gemm_f16's narrow shape (64 weight rows per block, 256 columns in flight per wave). It wins by
// the loads in flight, so by K; it loses by reading the token rows from L2 once per 16 rows, so by rows and tokens.
// Measured in us, narrow / few, at 1, 16 and 64 tokens:
//   K 256, 1026 rows 4.8 / 4.8, 4.9 / 4.8, 4.9 / 5.1; 9234 rows 4.8 / 4.8, 5.0 / 6.6, 6.3 / 10.5
//   K 512, 3078 rows 5.0 / 4.8, 5.9 / 4.9, 7.3 / 6.3; 4104 rows 4.9 / 4.8, 5.8 / 4.9, 7.5 / 8.4; 512 rows 4.0 / 3.9,
//          4.7 / 4.0, 4.7 / 5.3; 9234 rows 4.9 / 5.1, 6.2 / 7.2, 10.8 / 12.0
//   K 768, 9234 rows 6.1 / 5.4, 7.7 / 8.0, 14.1 / 14.0; 18468 rows 10.0 / 9.1, 11.0 / 13.6, 20.9 / 21.4
//   K 1024, 9234 rows 10.8 / 5.3, 12.3 / 8.4, 17.2 / 17.0; 18468 rows 12.9 / 10.6, 14.2 / 15.6, 25.7 / 25.4
//   K 1536, 18468 rows 19.3 / 13.6, 20.2 / 20.2, 35.4 / 32.9
//   K 2048, 18468 rows 24.4 / 17.0, 25.8 / 22.7, 45.4 / 39.7; 36864 rows 28.0 / 28.9, 30.2 / 39.2, 58.5 / 61.6
//   nsb: 256-column superblocks of K
inline bool f16_few_rows(int64_t rows, int nsb, int n_tok) {
    return nsb >= 2 && rows <= 4096ll * nsb && (nsb > 2 || n_tok <= 32);
}

// Q8_0 and Q6_K expert matmuls: the GEMMs instead of the GEMVs. From 8 routes per expert on average the GEMV reads its weights
// again for every 8 or 16 routes of an expert. A launch whose routes the GEMV blocks could list by themselves (`list` at
// most) pays another launch of about 4 us for the GEMM, the route sort: there the line follows the work saved, which grows with
// the routes and the weights of an expert (`elems` per matrix). Whole MoE layer calls, us, GEMV / GEMM, by routes:
//   Q8_0  512 x 256, 8 experts: 72 38.8 / 42.2, 512 42.8 / 43.8, 800 51.1 / 46.1; 1024 x 768, 16 experts: 192 47.6 / 49.1, 320
//         55.1 / 52.4; 2048 x 1536, 32 experts: 256 91.3 / 92.9 (Zipf 1.2: 78 / 62), 288 99.1 / 95.5; 4 experts: 64
//         48.1 / 49.0, 256 60.5 / 59.7; 16 experts: 256 65.5 / 68.9, 320 73.2 / 69.3
//   Q6_K  512 x 256, 8 experts: 72 40.0 / 42.6, 384 44.6 / 43.4; 1024 x 768, 8 experts: 72 45.0 / 46.9, 160 51.0 / 50.3;
//         2048 x 1536, 32 experts: 256 105 / 85; 4 experts: 64 56.4 / 53.5
inline bool quant_gemm_experts(bool q6_k, int64_t routes, int E, int64_t elems, int64_t list) {
    if (routes < 8ll * E) return false;
    const double work = (double) routes * (double) routes * (double) elems;
    return routes > list || (q6_k ? work >= 1.3e10 : routes >= 640 || work >= 1.6e11);
}

// The router down projection alone (an MoE layer call): k_router_down_t, which loads a weight row once for many tokens, instead
// of k_router_down's block per token and four outputs. Up to 512 columns it is never the slower one; above, it pays from
// about the work of 65 rows of 2048 columns, and rows of more than 2048 columns that leave part of the last chain step
// idle (d not 64 times a power of two) from 80 rows. us, per token / reusing,
// 128 outputs: d 512 at 128 rows 4.2 / 4.2, 256 6.5 / 4.2; d 768 at 65 4.2 / 5.7, 160 6.8 / 7.0, 200 8.0 / 6.5; d 1024 at
// 65 4.1 / 5.2, 128 6.2 / 5.8; d 1280 at 65 6.2 / 7.9, 96 7.7 / 8.1, 112 8.6 / 8.2; d 2048 at 65 6.6 / 5.4; d 3072
// at 65 14.4 / 16.0, 80 16.8 / 16.2; d 4096 at 65 10.8 / 8.6.
//   full: d is 64 times a power of two
inline bool router_down_reuse(int T, int d, bool full) {
    return (d <= 512 || (int64_t) T * d >= 65 * 2048) && T >= (d > 2048 && !full ? 80 : 65);
}

} // namespace z2r
