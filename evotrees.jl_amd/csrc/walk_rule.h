// Which trees on every row end in the walk of all rows.  Host code only.
#pragma once
#include <math.h>
#include <stddef.h>
#include <stdint.h>

// Whether the rows of a tree on every row are walked through it at the end, in row order and with the next gradients computed on the way (k_predict_tree), or
// leave their leaf's number from its last level's lists, a scattered word each, for the gradient pass to look up.  The walk reads a line of a column
// for 128 rows where any of them tests that feature: of 128 rows at most min(2^l, 128) nodes of level l, of an oblivious tree one feature a level.  It is one kernel for two and shorter
// wherever the bins come from the caches, or fewer than about 88 bytes a row from memory; us a round, walk less than words: 60k to 1M rows of 20 to 100 features, depth 5 to 10, -1 to
// -30; 4M x 20 -19 to -51; 10M x 100, depth 6 (27 bytes) -58, 8 (72) -131, 11 (99) +59; 4M x 100, depth 11 +11; 10M x 20, depth 11 -162;
// 10M x 50 of two outputs, depth 11 (50) -121; oblivious, 10M x 100, depth 9 (8 bytes) -82, 11 (10) -52, 4M x 100, depth 8 -25, 11 -16.
static inline bool walk_pays(int64_t rows, int all_feats, int feats, int depth, bool oblivious) {
    if ((size_t)rows * all_feats <= (size_t)256 << 20) return true; // what the last-level cache holds
    double nodes = 0;
    for (int l = 0; l + 1 < depth; l++) nodes += oblivious ? 1 : l < 7 ? 1 << l : 128;
    return feats * (1 - exp(-nodes / feats)) <= 88;
}
