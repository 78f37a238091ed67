// Chunk depth of the Merkle stage kernels: a wave hashes 2^c chunks of 128
// items, merging them as it goes, and ends with a reduction of its last 64 nodes
// on narrow levels, to the one node 7 + c levels above its items or, in a large
// leaf stage, to the several nodes (`keep`) below it.
// Pure host logic (no device code), shared by the tree driver and its
// autotuner.
#pragma once
#include <stdint.h>

#include <atomic>

namespace vx {

constexpr uint32_t MERKLE_LOGC_MAX = 5;       // chunks per wave in a stage: up to 32
constexpr uint32_t STAGE_MIN_WAVES = 3072;    // pick_logc's own rule: three waves per SIMD
constexpr uint32_t STAGE_PLAN_LOGS = 40;      // table index: log2 of the items of one launch

// Tuned depth per log2 of the items one stage launch covers (every proof of a
// batch), stored as c + 1 (0: not tuned, use the default rule).
inline std::atomic<uint8_t>* stage_plan_table() {
    static std::atomic<uint8_t> t[STAGE_PLAN_LOGS];
    return t;
}

inline uint32_t floor_log2(uint64_t x) { return x ? 63u - (uint32_t)__builtin_clzll(x) : 0u; }

// Depth of a stage over n items per proof for `batch` proofs: the tuned depth
// for n * batch items when there is one and use_plan is set, else the largest
// c that still leaves STAGE_MIN_WAVES waves in the launch; never above
// logc_max, and always at least two waves per proof. Launches take their shape
// from pick_stage below, which comes here for tuned sizes alone and has a
// measured default of its own.
inline uint32_t pick_logc(uint64_t n, uint32_t logc_max = MERKLE_LOGC_MAX, uint32_t batch = 1, bool use_plan = true) {
    const uint32_t lt = floor_log2(n * batch);
    int c = use_plan && lt < STAGE_PLAN_LOGS ? (int)stage_plan_table()[lt].load(std::memory_order_relaxed) - 1 : -1;
    if (c < 0) {
        c = 0;
        for (int k = (int)logc_max; k > 0; k--) {
            const uint64_t w = n >> (7 + k);
            if (w >= 2 && w * batch >= STAGE_MIN_WAVES) {
                c = k;
                break;
            }
        }
    }
    if (c > (int)logc_max) c = (int)logc_max;
    while (c > 0 && (n >> (7 + c)) < 2) c--;
    return (uint32_t)c;
}

// What a stage wave does: 2^logc chunks of 128 items, handing on `keep` nodes.
struct StageShape {
    uint32_t logc, keep;
};

// Shape of a stage over n items per proof for `batch` proofs.
//
// A wave's LDS (a slot of 2 KiB per pending level) decides how many waves share
// a SIMD, and since a second wave's adds and xors issue beside the first one's
// rotations, more waves hash faster until about five share it (66-68 G
// compressions/s at 4-8 waves, 58 at 3). Shallow waves also fill the device
// sooner, but spend more of their life in the 64 -> 1 reduction, whose last
// levels leave most quads idle; so from 2^18 items a launch on, leaf waves
// hand on several nodes and the node stages compute the levels above, one node
// per lane. Whole quotient-tree commitments (us) on one MI355X, depth/keep:
//   2^17: 0/1 34, 1/1 39           2^20: 0/1 90, 1/16 76, 2/1 77, 2/16 73
//   2^22: 2/1 193, 2/16 185, 3/16 184, 4/16 189
//   2^24: 2/16 612, 3/1 613, 3/16 602, 5/1 633
//   2^26: 2/16 2311, 3/16 2268, 4/1 2276, 4/16 2245, 5/1 2267
// (2^26 ran at 5/16 with one more slot a wave before: 2382 for the leaf stage
// alone.) Node trees: 2^17 nodes 0: 30, 1: 31; 2^18 0: 40, 1: 35; 2^19 1: 46,
// 2: 44; so a node launch takes the depth of a leaf launch twice its size.
inline StageShape pick_stage(uint64_t n, uint32_t logc_max, uint32_t batch, bool use_plan, bool nodes) {
    const uint32_t lt = floor_log2(n * batch);
    const bool tuned = use_plan && lt < STAGE_PLAN_LOGS && stage_plan_table()[lt].load(std::memory_order_relaxed) != 0;
    uint32_t c;
    if (tuned) {
        c = pick_logc(n, logc_max, batch);
    } else {
        const uint32_t l = lt + (nodes ? 1 : 0);
        c = l >= 25 ? 4 : l >= 22 ? 3 : l >= 20 ? 2 : l >= 19 ? 1 : 0;
        if (c > logc_max) c = logc_max;
        while (c > 0 && (n >> (7 + c)) < 2) c--;
    }
    // at most n / 32 nodes whatever the depth (max_leaf_stage_nodes)
    uint32_t keep = 1;
    if (!nodes && lt >= 18) keep = c >= 2 ? 16 : 4u << c;
    return {c, keep};
}

// Most nodes a leaf stage of a tree of n_leaves items hands on (per proof).
inline uint64_t max_leaf_stage_nodes(uint64_t n_leaves, uint64_t tail_items) {
    return n_leaves <= tail_items ? 0 : n_leaves >> 5;
}
// Most nodes any stage of a tree of n_leaves items that hands on one node a
// wave can output (per proof), whatever depth is picked: a wave covers at
// least 128 items.
inline uint64_t max_stage_nodes(uint64_t n_leaves, uint64_t tail_items) {
    return n_leaves <= tail_items ? 0 : n_leaves >> 7;
}

}  // namespace vx
