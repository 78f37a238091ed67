// Host-side driver of the Merkle engine: commits a leaf source with one stage
// kernel over the leaves, stage kernels over node layers while more than
// PROVER_TAIL_ITEMS nodes remain, and the tail kernel (root + transcript).
#pragma once
#include <algorithm>

#include "common.hpp"
#include "merkle_engine.hpp"

namespace vx {

// Trees of at most this many items go straight to the tail kernel; larger
// ones are reduced by stage kernels until this many nodes remain (one more
// tail level is cheaper than one more stage launch).
constexpr uint32_t PROVER_TAIL_ITEMS = MERKLE_TAIL_MAX;

// Leaf trees of at most this many leaves are one tail launch; larger ones spread
// their leaves over many CUs first.
constexpr uint32_t QUAD_DIRECT_MAX = 1024;

struct Scratch {
    uint32_t* a;
    uint32_t* b;
};

// Commits n_leaves (power of two >= 2) items of a leaf source, for `batch`
// proofs at once whose buffers are bs words apart (bs = 0 for one proof).
// Trees of at most direct_max leaves go straight to the tail kernel.
template <class Src, class Mark>
void commit_tree(const Src& src, uint64_t n_leaves, LevelStore st, TailOut out, Scratch sc, hipStream_t s,
                 Mark&& mark, uint32_t batch = 1, uint64_t bs = 0, uint64_t direct_max = PROVER_TAIL_ITEMS) {
    if (n_leaves <= direct_max) {
        launch_tail(src, 0, (uint32_t)n_leaves, st, out, batch, bs, s);
        check_launch("merkle_tail_kernel");
        mark("tail");
        return;
    }
    auto grid = [&](uint64_t waves) { return dim3(ceil_div(waves, MERKLE_STAGE_WAVES), batch); };
    StageShape sh = pick_stage(n_leaves, StageLogcMax<Src>::value, batch, stage_uses_plan<Src>(), false);
    uint64_t waves = n_leaves >> (7 + sh.logc);
    merkle_stage_kernel<Src><<<grid(waves), 64 * MERKLE_STAGE_WAVES, stage_lds_bytes(sh.logc), s>>>(
        src, 0, n_leaves, sh.logc, sc.a, st, bs, sh.keep);
    check_launch("merkle_stage_kernel");
    mark("stage_leaf");
    uint64_t n = waves * sh.keep;
    uint32_t lvl = 7 + sh.logc - floor_log2(sh.keep);
    uint32_t* cur = sc.a;
    uint32_t* nxt = sc.b;
    while (n > PROVER_TAIL_ITEMS) {
        sh = pick_stage(n, MERKLE_LOGC_MAX, batch, true, true);
        waves = n >> (7 + sh.logc);
        merkle_stage_kernel<SrcNodes><<<grid(waves), 64 * MERKLE_STAGE_WAVES, stage_lds_bytes(sh.logc), s>>>(
            SrcNodes{cur}, lvl, n, sh.logc, nxt, st, bs, sh.keep);
        check_launch("merkle_stage_kernel<nodes>");
        mark("stage_node");
        n = waves;
        lvl += 7 + sh.logc;
        uint32_t* tmp = cur;
        cur = nxt;
        nxt = tmp;
    }
    launch_tail(SrcNodes{cur}, lvl, (uint32_t)n, st, out, batch, bs, s);
    check_launch("merkle_tail_kernel<nodes>");
    mark("tail");
}

// Trees of at most LEAF_QUAD_MAX leaves (and more than a tail kernel should
// hash by itself) of a single proof commit through leaf_quad_stage_kernel, 16
// leaves a wave up to 2^14 leaves, 32 at 2^15, 64 at 2^16, so the tail starts
// from at most 256 nodes, all of whose levels go by quads. Such a tree's chain is
// latency-bound for one proof (2^14 rows: 292 us with 512 nodes handed on and the
// line at 2^15, 274 so; the line at 2^17 is 1 % slower from 2^15 rows on); a batch
// of proofs fills the device with its waves, where the lane-per-pair stage does
// the same hashing in fewer instructions (about 980 a compression against 4 x
// 390), so batches keep it.
constexpr uint64_t LEAF_QUAD_MAX = 1ull << 16;
inline uint32_t quad_stage_leaves(uint64_t n) { return n <= (1ull << 14) ? 16u : n <= (1ull << 15) ? 32u : 64u; }

// Commits a tree of n leaves (1024 <= n <= LEAF_QUAD_MAX, a power of two) with
// the quad leaf stage and the tail kernel. Its stage hands on n / 64 nodes at
// most (scratch_nodes_a).
template <class Src, class Mark>
void commit_tree_quad(const Src& src, uint64_t n, LevelStore st, TailOut out, Scratch sc, hipStream_t s, Mark&& mark,
                      uint32_t batch = 1, uint64_t bs = 0) {
    const uint32_t lpw = quad_stage_leaves(n);
    const uint32_t blocks = (uint32_t)(n / (lpw * LEAF_QUAD_WAVES));
    const dim3 grid(blocks, batch);
    if (lpw == 16)
        leaf_quad_stage_kernel<Src, 1><<<grid, 64 * LEAF_QUAD_WAVES, 0, s>>>(src, sc.a, st, bs);
    else if (lpw == 32)
        leaf_quad_stage_kernel<Src, 2><<<grid, 64 * LEAF_QUAD_WAVES, 0, s>>>(src, sc.a, st, bs);
    else
        leaf_quad_stage_kernel<Src, 4><<<grid, 64 * LEAF_QUAD_WAVES, 0, s>>>(src, sc.a, st, bs);
    check_launch("leaf_quad_stage_kernel");
    mark("stage_leaf");
    launch_tail(SrcNodes{sc.a}, floor_log2(lpw * LEAF_QUAD_WAVES), blocks, st, out, batch, bs, s);
    check_launch("merkle_tail_kernel<nodes>");
    mark("tail");
}

// A tree of a prover: by quads for a single proof's small trees, by commit_tree
// otherwise; trees of at most direct_max leaves are one tail launch.
template <class Src, class Mark>
void commit_leaves(const Src& src, uint64_t n, LevelStore st, TailOut out, Scratch sc, hipStream_t s, Mark&& mark,
                   uint32_t batch, uint64_t bs) {
    if (batch == 1 && n > QUAD_DIRECT_MAX && n <= LEAF_QUAD_MAX)
        commit_tree_quad(src, n, st, out, sc, s, mark, batch, bs);
    else
        commit_tree(src, n, st, out, sc, s, mark, batch, bs, QUAD_DIRECT_MAX);
}

// Nodes per proof of the two stage scratch buffers of a tree of n_leaves items:
// a takes the leaf stage's output and every other node stage's, b the rest.
inline uint64_t scratch_nodes_a(uint64_t n_leaves) {
    const uint64_t quad = n_leaves <= QUAD_DIRECT_MAX ? 0 : std::min<uint64_t>(n_leaves, LEAF_QUAD_MAX) / (16 * LEAF_QUAD_WAVES);
    return std::max<uint64_t>({1, max_leaf_stage_nodes(n_leaves, QUAD_DIRECT_MAX), quad});
}
inline uint64_t scratch_nodes_b(uint64_t n_leaves) {
    return std::max<uint64_t>(1, max_stage_nodes(scratch_nodes_a(n_leaves), 0));
}

}  // namespace vx
