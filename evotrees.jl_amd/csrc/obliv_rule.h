// Which oblivious levels k_obliv_level decides in one launch: its instances and the rule that chooses it, in one place, so that the rule admits
// no level without an instance.  Host code only.
#pragma once

#define OBLIV_LEVEL_NODES 32
// the kernel's instances: accumulator channels, bins of a lane, nodes of a wavefront
#define EVT_OBLIV_LEVELS(X)                                                                                     \
    X(2, 1, 1) X(2, 2, 1) X(2, 4, 1) X(3, 1, 1) X(3, 2, 1) X(3, 4, 1) X(5, 1, 1) X(5, 2, 1) X(5, 4, 1) \
    X(2, 1, 2) X(2, 2, 2) X(2, 4, 2) X(3, 1, 2) X(3, 2, 2) X(5, 1, 2)

// a lane's bins as the instances have them
inline int obliv_lane_bins(int bins) { return bins <= 64 ? 1 : bins <= 128 ? 2 : 4; }
inline int obliv_wave_nodes(int nodes) { return nodes > 16 ? 2 : 1; }

// Where a wavefront's words (nodes x channels x 64-bin pieces) are few enough for its registers and the searches a block's wavefronts share do not
// outlast the launches saved.  us of a level in three launches | one, event pairs included (60k rows; 20 to 120
// features): mse 64 bins 4 nodes 14 | 8, 16 nodes 16 | 9, 32 nodes 19 | 14; mse 128 bins 32 nodes 21 | 19; mse 255 bins 16 nodes 20 | 18, 32 nodes 27 | 32;
// logloss 128 bins 16 nodes 18 | 13, 32 nodes 21 | 21; two outputs 64 bins 16 nodes 14 | 13, 128 bins 16 nodes 17 | 17, 255 bins 8 nodes 25 | 20, 16 nodes 24 | 32.
// Whole rounds of depth 7, mse of 160 bins, the level of 32 nodes in three launches | one: 60k x 20 135 | 130, 60k x 120 145 | 141, 500k x 50 189 | 183.
inline bool obliv_level_fits(int channels, int bins, int nodes) {
    if (bins < 4 || nodes > OBLIV_LEVEL_NODES || nodes * channels * ((bins + 63) / 64) > 192) return false;
#define EVT_HAS(NAG_, BPL_, NPW_) \
    if (channels == NAG_ && obliv_lane_bins(bins) == BPL_ && obliv_wave_nodes(nodes) == NPW_) return true;
    EVT_OBLIV_LEVELS(EVT_HAS)
#undef EVT_HAS
    return false;
}
