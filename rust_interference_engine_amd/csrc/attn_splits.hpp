// attn_splits.hpp — KV splits of the prompt attention (host code without HIP).
#pragma once

#include <algorithm>

namespace rie {

// Splits of a prompt attention launch of wgs workgroups whose longest query row sees
// `tiles` tiles of 32 positions; a second kernel merges them.
// * From 64 workgroups on: splits of at least 16 tiles, up to about two workgroups per CU
//   (finer ones, by the rule below, measured no better: at 0 / at 800, two layers of 64
//   workgroups 733 / 744 against 726 / 750 us, 88 508 / 527 against 500 / 528, 96 503 / 491
//   against 501 / 493, 112 1100 / 1123 against 1098 / 1122; 128 at 0 1149 against 1142).
// * Below: splits of at least 2 tiles, up to one workgroup per CU (650 tokens of
//   gemma-3-1b, 21 workgroups, six layers: 1579 us in one pass with the per-token kernel,
//   1369 us in splits of 4 tiles, 1323 us in splits of 2; two workgroups per CU are slower
//   on long rows too: 128 tokens at 15000, 32 workgroups of two layers, 16 splits 660 us
//   against 624 us with 8, Q8_0 cache 739 against 696 us).
// * At most 16, and 32 over Q8_0 caches, where the per-token kernel that ran these calls
//   before had 32 ranges (2 tokens at 12000, 8 workgroups: 308 us with 16, 281 us with 32,
//   290 us in that kernel).
inline int prompt_kv_splits(int wgs, int tiles, bool q8_0) {
    const int s = wgs < 64 ? std::min(tiles / 2, 256 / wgs) : std::min(tiles / 16, 512 / wgs);
    return std::max(1, std::min(q8_0 ? 32 : 16, s));
}

}  // namespace rie
