// Wave64 Blake2s Merkle engine with fused leaf producers.
//
// Tree semantics are the reference's (src/merkle.rs:28-104, cuda/blake2s.cu):
// complete binary tree, leaf = Blake2s(LE32 words), parent = Blake2s(L || R),
// no personalisation. What differs is the execution model:
//
//  * A "source" produces the items of one tree level. Leaf sources hash data
//    (one M31 column, four SoA columns, the Fibonacci quotient computed on the
//    fly from the LDE, or an FRI circle/line fold computed and stored on the
//    fly); the node source reads 8-word hashes produced by a previous kernel.
//  * Stage kernel: every wave owns 128 * 2^logc consecutive items. Each step
//    the 64 lanes compute 64 parents of 128 items (one chunk); chunks merge
//    pairwise like a binary counter, the left chunk waiting in the wave's LDS
//    stack, so every compression runs with all 64 lanes busy and no
//    workgroup barrier is ever needed. The last 64 nodes are reduced with
//    quad-cooperative compressions (4 lanes each): to one, 7 + logc levels above
//    the wave's items, or in large leaf stages to the 4 to 16 nodes where quads
//    would leave most lanes idle, which the next stage hashes one per lane.
//  * Small trees of a single proof: a quad per leaf, one node a workgroup.
//  * Tail kernel: one workgroup reduces the last <= 2048 items to the root,
//    writes it where the caller asks and advances the Fiat-Shamir transcript
//    (mix the root, draw the next challenge) in the same launch; its narrow
//    levels and the transcript hashes also run quad-cooperatively.
//  * Every node at level >= store_from is also written to a per-tree level
//    store; decommitment recomputes the 2^store_from-leaf subtree of a query
//    and reads the rest, so full trees are never written to HBM.
#pragma once
#include <type_traits>

#include "stage_plan.hpp"
#include "blake2s.hpp"
#include "field.hpp"
#include "transcript.hpp"

namespace vx {

// Orders this wave's LDS writes before its later LDS reads (the LDS executes a
// wave's requests in order; this keeps the compiler from reordering them).
#define VX_WAVE_SYNC()                                        \
    do {                                                      \
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); \
        __builtin_amdgcn_wave_barrier();                      \
    } while (0)

constexpr uint32_t MERKLE_TAIL_MAX = 2048;  // most items one tail-kernel block reduces
constexpr uint32_t MERKLE_STAGE_WAVES = 4;  // waves per stage workgroup

// Nodes of levels [from, depth] of a tree with 2^depth leaves, level-major.
struct LevelStore {
    uint32_t* base;
    uint32_t depth;
    uint32_t from;
    __device__ __forceinline__ bool want(uint32_t level) const { return base && level >= from && level <= depth; }
    __device__ __forceinline__ uint32_t* at(uint32_t level, uint64_t idx) const {
        uint64_t off = (1ull << (depth - from + 1)) - (1ull << (depth - level + 1));
        return base + 8ull * (off + idx);
    }
    __device__ __forceinline__ LevelStore shifted(uint64_t off) const {
        return {base ? base + off : nullptr, depth, from};
    }
};
__host__ __device__ inline uint64_t level_store_words(uint32_t depth, uint32_t from) {
    return from > depth ? 0 : 8ull * ((1ull << (depth - from + 1)) - 1);
}

__device__ __forceinline__ void store8(uint32_t* dst, const uint32_t h[8]) {
    uint4* d = (uint4*)dst;
    d[0] = make_uint4(h[0], h[1], h[2], h[3]);
    d[1] = make_uint4(h[4], h[5], h[6], h[7]);
}
__device__ __forceinline__ void load8(const uint32_t* src, uint32_t h[8]) {
    const uint4* s = (const uint4*)src;
    uint4 a = s[0], b = s[1];
    h[0] = a.x;
    h[1] = a.y;
    h[2] = a.z;
    h[3] = a.w;
    h[4] = b.x;
    h[5] = b.y;
    h[6] = b.z;
    h[7] = b.w;
}

// Parent of the SoA4 leaves of two QM31 values.
template <bool PRIO>
__device__ __forceinline__ void b2s_leaf_pair4(const QM31& x, const QM31& y, uint32_t h[8]) {
    const uint32_t w[2][4] = {{x.v[0], x.v[1], x.v[2], x.v[3]}, {y.v[0], y.v[1], y.v[2], y.v[3]}};
    b2s_leaf_pair<4, PRIO>(w, h);
}

// ---------------------------------------------------------------- sources
// pair(i, h): i even; h = parent of items i and i+1.
// leaf(i, h) / values(i, v): used by decommitment (leaf sources only).
// at(off): the same source for another proof of a batch, whose buffers sit
// `off` words further (batched provers give every proof an equal-size arena;
// shared tables such as twiddles do not move).

// words(i, l, v): the WIDTH words of leaf i, for a quad whose four lanes all call
// it; a source that stores what it forms stores coordinate l.

struct SrcNodes {
    const uint32_t* nodes;
    __device__ __forceinline__ SrcNodes at(uint64_t off) const { return {nodes + off}; }
    template <bool PRIO = true>
    __device__ __forceinline__ void pair(uint64_t i, uint32_t h[8]) const {
        uint32_t l[8], r[8];
        load8(nodes + 8 * i, l);
        load8(nodes + 8 * i + 8, r);
        b2s_node(l, r, h);
    }
};

// One M31 column (the trace LDE); leaf = H(LE32(v)), t = 4.
struct SrcCol1 {
    const uint32_t* col;
    static constexpr uint32_t WIDTH = 1;
    __device__ __forceinline__ SrcCol1 at(uint64_t off) const { return {col + off}; }
    __device__ __forceinline__ void values(uint64_t i, uint32_t v[4]) const { v[0] = col[i]; }
    __device__ __forceinline__ void words(uint64_t i, uint32_t, uint32_t v[1]) const { v[0] = col[i]; }
    __device__ __forceinline__ void leaf(uint64_t i, uint32_t h[8]) const { b2s_leaf1(col[i], h); }
    template <bool PRIO = true>
    __device__ __forceinline__ void pair(uint64_t i, uint32_t h[8]) const {
        uint2 v = *(const uint2*)(col + i);
        const uint32_t w[2][1] = {{v.x}, {v.y}};
        b2s_leaf_pair<1, PRIO>(w, h);
    }
};

// Four SoA columns (a QM31 column); leaf = H(16 bytes), t = 16.
struct SrcSoa4 {
    const uint32_t* c0;
    const uint32_t* c1;
    const uint32_t* c2;
    const uint32_t* c3;
    static constexpr uint32_t WIDTH = 4;
    __device__ __forceinline__ SrcSoa4 at(uint64_t off) const { return {c0 + off, c1 + off, c2 + off, c3 + off}; }
    __device__ __forceinline__ void values(uint64_t i, uint32_t v[4]) const {
        v[0] = c0[i];
        v[1] = c1[i];
        v[2] = c2[i];
        v[3] = c3[i];
    }
    __device__ __forceinline__ void leaf(uint64_t i, uint32_t h[8]) const {
        b2s_leaf4(c0[i], c1[i], c2[i], c3[i], h);
    }
    template <bool PRIO = true>
    __device__ __forceinline__ void pair(uint64_t i, uint32_t h[8]) const {
        uint2 a = *(const uint2*)(c0 + i), b = *(const uint2*)(c1 + i);
        uint2 c = *(const uint2*)(c2 + i), d = *(const uint2*)(c3 + i);
        const uint32_t w[2][4] = {{a.x, b.x, c.x, d.x}, {a.y, b.y, c.y, d.y}};
        b2s_leaf_pair<4, PRIO>(w, h);
    }
};

// Fibonacci quotient evaluated on the fly from the LDE t (size mask+1):
// q[i] = alpha * (t[i+2] - (t[i+1] + t[i])), indices mod E (constraint.cu:10-36).
__device__ __forceinline__ QM31 quotient_at(uint32_t t0, uint32_t t1, uint32_t t2, QM31 alpha) {
    return qmul_m31(alpha, msub(t2, madd(t1, t0)));
}
// A challenge, written by an earlier launch: the same four words for every lane,
// so they come by scalar loads.
__device__ __forceinline__ QM31 load_alpha(const uint32_t* a) {
    ConstU32* c = (ConstU32*)a;
    return {{c[0], c[1], c[2], c[3]}};
}

struct SrcQuotient {
    const uint32_t* t;
    uint64_t mask;
    const uint32_t* alpha;  // device, 4 words
    static constexpr uint32_t WIDTH = 4;
    __device__ __forceinline__ SrcQuotient at(uint64_t off) const { return {t + off, mask, alpha + off}; }
    __device__ __forceinline__ QM31 q(uint64_t i, QM31 al) const {
        return quotient_at(t[i], t[(i + 1) & mask], t[(i + 2) & mask], al);
    }
    __device__ __forceinline__ void values(uint64_t i, uint32_t v[4]) const {
        QM31 r = q(i, load_alpha(alpha));
        for (int k = 0; k < 4; k++) v[k] = r.v[k];
    }
    __device__ __forceinline__ void words(uint64_t i, uint32_t, uint32_t v[4]) const { values(i, v); }
    __device__ __forceinline__ void leaf(uint64_t i, uint32_t h[8]) const {
        QM31 r = q(i, load_alpha(alpha));
        b2s_leaf4(r.v[0], r.v[1], r.v[2], r.v[3], h);
    }
    template <bool PRIO = true>
    __device__ __forceinline__ void pair(uint64_t i, uint32_t h[8]) const {
        QM31 al = load_alpha(alpha);
        uint2 a = *(const uint2*)(t + i);
        uint2 b = *(const uint2*)(t + ((i + 2) & mask));
        QM31 q0 = quotient_at(a.x, a.y, b.x, al);
        QM31 q1 = quotient_at(a.y, b.x, b.y, al);
        b2s_leaf_pair4<PRIO>(q0, q1, h);
    }
};

// First FRI layer: circle fold of the quotient (recomputed from the LDE),
// stored to out and hashed (fri.cu:44-78 with a zero-initialised destination,
// so the layer equals the fold f' itself).
struct SrcCircleFold {
    const uint32_t* t;
    uint64_t mask;
    const uint32_t* alpha_q;
    const uint32_t* alpha_f;
    const uint32_t* tw;
    uint32_t* o0;
    uint32_t* o1;
    uint32_t* o2;
    uint32_t* o3;
    __device__ __forceinline__ SrcCircleFold at(uint64_t off) const {
        return {t + off, mask, alpha_q + off, alpha_f + off, tw, o0 + off, o1 + off, o2 + off, o3 + off};
    }
    // With q(i) = aq * d(i), d(i) = t[i+2] - t[i+1] - t[i] an M31 value, the fold
    // (q0 + q1) + af * ((q0 - q1) * tw) equals aq * (d0 + d1) + (af * aq) * ((d0 - d1) * tw):
    // nine M31 products and five reductions per output.
    __device__ __forceinline__ static QM31 fold_d(uint32_t d0, uint32_t d1, QM31 aq, QM31 g, uint32_t tw) {
        const uint32_t s = madd(d0, d1), u = mmul(msub(d0, d1), tw);
        QM31 r;
#pragma unroll
        for (int k = 0; k < 4; k++) r.v[k] = reduce64((uint64_t)aq.v[k] * s + (uint64_t)g.v[k] * u);
        return r;
    }
    static constexpr uint32_t WIDTH = 4;
    __device__ __forceinline__ void words(uint64_t i, uint32_t l, uint32_t v[4]) const {
        const QM31 aq = load_alpha(alpha_q), g = qmul(load_alpha(alpha_f), aq);
        const uint64_t j = 2 * i;
        const uint2 a = *(const uint2*)(t + j);
        const uint2 b = *(const uint2*)(t + ((j + 2) & mask));
        const QM31 f = fold_d(msub(b.x, madd(a.y, a.x)), msub(b.y, madd(b.x, a.y)), aq, g, tw[i]);
        for (int k = 0; k < 4; k++) v[k] = f.v[k];
        store_coord(i, l, f);
    }
    __device__ __forceinline__ void store_coord(uint64_t i, uint32_t l, const QM31& f) const {
        uint32_t* o = l == 0 ? o0 : l == 1 ? o1 : l == 2 ? o2 : o3;
        o[i] = l == 0 ? f.v[0] : l == 1 ? f.v[1] : l == 2 ? f.v[2] : f.v[3];
    }
    template <bool PRIO = true>
    __device__ __forceinline__ void pair(uint64_t i, uint32_t h[8]) const {
        const QM31 aq = load_alpha(alpha_q), g = qmul(load_alpha(alpha_f), aq);
        uint64_t j = 2 * i;  // quotient index of the first of four inputs
        uint2 a = *(const uint2*)(t + j);
        uint2 b = *(const uint2*)(t + ((j + 2) & mask));
        uint2 c = *(const uint2*)(t + ((j + 4) & mask));
        uint2 w = *(const uint2*)(tw + i);
        const uint32_t d0 = msub(b.x, madd(a.y, a.x)), d1 = msub(b.y, madd(b.x, a.y));
        const uint32_t d2 = msub(c.x, madd(b.y, b.x)), d3 = msub(c.y, madd(c.x, b.y));
        QM31 f0 = fold_d(d0, d1, aq, g, w.x);
        QM31 f1 = fold_d(d2, d3, aq, g, w.y);
        *(uint2*)(o0 + i) = make_uint2(f0.v[0], f1.v[0]);
        *(uint2*)(o1 + i) = make_uint2(f0.v[1], f1.v[1]);
        *(uint2*)(o2 + i) = make_uint2(f0.v[2], f1.v[2]);
        *(uint2*)(o3 + i) = make_uint2(f0.v[3], f1.v[3]);
        b2s_leaf_pair4<PRIO>(f0, f1, h);
    }
};

// Line fold of the previous layer, stored to out and hashed (fri.cu:10-39).
struct SrcLineFold {
    const uint32_t* i0;
    const uint32_t* i1;
    const uint32_t* i2;
    const uint32_t* i3;
    const uint32_t* alpha;
    const uint32_t* tw;
    uint32_t* o0;
    uint32_t* o1;
    uint32_t* o2;
    uint32_t* o3;
    __device__ __forceinline__ SrcLineFold at(uint64_t off) const {
        return {i0 + off, i1 + off, i2 + off, i3 + off, alpha + off, tw, o0 + off, o1 + off, o2 + off, o3 + off};
    }
    static constexpr uint32_t WIDTH = 4;
    __device__ __forceinline__ void words(uint64_t i, uint32_t l, uint32_t v[4]) const {
        const uint2 a = *(const uint2*)(i0 + 2 * i), b = *(const uint2*)(i1 + 2 * i);
        const uint2 c = *(const uint2*)(i2 + 2 * i), d = *(const uint2*)(i3 + 2 * i);
        const QM31 f = fold_pair({{a.x, b.x, c.x, d.x}}, {{a.y, b.y, c.y, d.y}}, QMatrix(load_alpha(alpha)), tw[i]);
        for (int k = 0; k < 4; k++) v[k] = f.v[k];
        uint32_t* o = l == 0 ? o0 : l == 1 ? o1 : l == 2 ? o2 : o3;
        o[i] = l == 0 ? f.v[0] : l == 1 ? f.v[1] : l == 2 ? f.v[2] : f.v[3];
    }
    template <bool PRIO = true>
    __device__ __forceinline__ void pair(uint64_t i, uint32_t h[8]) const {
        const QMatrix al(load_alpha(alpha));
        uint64_t j = 2 * i;
        uint4 a = *(const uint4*)(i0 + j), b = *(const uint4*)(i1 + j);
        uint4 c = *(const uint4*)(i2 + j), d = *(const uint4*)(i3 + j);
        uint2 w = *(const uint2*)(tw + i);
        QM31 f0 = fold_pair({{a.x, b.x, c.x, d.x}}, {{a.y, b.y, c.y, d.y}}, al, w.x);
        QM31 f1 = fold_pair({{a.z, b.z, c.z, d.z}}, {{a.w, b.w, c.w, d.w}}, al, w.y);
        *(uint2*)(o0 + i) = make_uint2(f0.v[0], f1.v[0]);
        *(uint2*)(o1 + i) = make_uint2(f0.v[1], f1.v[1]);
        *(uint2*)(o2 + i) = make_uint2(f0.v[2], f1.v[2]);
        *(uint2*)(o3 + i) = make_uint2(f0.v[3], f1.v[3]);
        b2s_leaf_pair4<PRIO>(f0, f1, h);
    }
};

// Lifted multi-column leaves (cuda/merkle_leaves_lifted.cu:26-98): leaf i hashes,
// with standard streaming Blake2s (full blocks non-final, the last block final,
// t = bytes so far), the LE32 words of every column in the given order, column
// c read at row i when its log size equals the tree's, else at
// ((i >> sh) << 1) | (i & 1) with sh = S - log_size + 1.
struct LiftCol {
    const uint32_t* p;
    uint32_t sh;  // 0: full-size column
    uint32_t pad;
};
// The column table is read-only for the whole launch and every lane reads the
// same entry: reading it through the constant address space lets the compiler
// use scalar loads, and the column data through the global one plain vector
// loads (a generic pointer would make them flat loads).
typedef const __attribute__((address_space(4))) LiftCol ConstLiftCol;
typedef const gu32x2 GlobalV2;
typedef const gu32x4 GlobalV4;
__device__ __forceinline__ ConstLiftCol* const_table(const LiftCol* t) { return (ConstLiftCol*)t; }

struct SrcLifted {
    static constexpr uint32_t STAGE_LOGC_MAX = 2;  // 2^22 leaves: depth 1 312 us, 2 306, 3 323, 4 374
    const LiftCol* cols;  // device, hashing order
    uint32_t n_cols;
    __device__ __forceinline__ SrcLifted at(uint64_t) const { return *this; }
    // leaves i (even) and i + 1 read rows r and r + 1 of every column
    __device__ __forceinline__ void load_block(ConstLiftCol* tab, uint32_t c0, uint64_t i, uint2 v[16]) const {
        const uint32_t nw = n_cols - c0 < 16 ? n_cols - c0 : 16;
#pragma unroll
        for (uint32_t k = 0; k < 16; k++) {
            v[k] = make_uint2(0, 0);
            if (k < nw) {
                const uint32_t* p = tab[c0 + k].p;
                const uint32_t sh = tab[c0 + k].sh;
                const uint64_t r = sh ? ((i >> sh) << 1) : i;
                const u32x2 x = *(GlobalV2*)(p + r);
                v[k] = make_uint2(x.x, x.y);
            }
        }
    }
    // One block's loads at a time: holding the next block's 32 words as well
    // (to have them in flight while this one is hashed) costs 146 VGPRs, three
    // waves a SIMD; without them four waves share it (98) and cover each other's
    // loads, and the hashing itself pairs better (34 columns, 2^22 leaves:
    // 368 -> 306 us).
    template <bool PRIO = true>
    __device__ __forceinline__ void pair(uint64_t i, uint32_t h[8]) const {
        ConstLiftCol* tab = const_table(cols);
        uint32_t ha[8], hb[8];
        b2s_init(ha);
        b2s_init(hb);
        for (uint32_t c0 = 0;; c0 += 16) {
            const bool last = c0 + 16 >= n_cols;
            uint2 v[16];
            load_block(tab, c0, i, v);
            uint32_t ma[16], mb[16];
#pragma unroll
            for (uint32_t k = 0; k < 16; k++) {
                ma[k] = v[k].x;
                mb[k] = v[k].y;
            }
            const uint32_t nw = n_cols - c0 < 16 ? n_cols - c0 : 16;
            const uint32_t t = 4 * (c0 + nw), f = last ? 0xFFFFFFFFu : 0u;
            b2s_compress<16, PRIO>(ha, ma, t, f);
            b2s_compress<16, PRIO>(hb, mb, t, f);
            if (last) break;
        }
        b2s_node<PRIO>(ha, hb, h);
    }
};

// First FRI layer of the wide commitment: f = sum_c beta^c * lifted_c is formed
// on the fly from the LDE columns, circle-folded pairwise (2j, 2j + 1) with
// alpha and tw[j], stored to out and hashed as an SoA4 leaf.
struct SrcWideFold {
    static constexpr uint32_t STAGE_LOGC_MAX = 2;  // 2^21 leaves: depth 1 170 us, 2 180, 3 213
    const LiftCol* cols;  // ascending in size: the lifted columns come before the full-size ones
    uint32_t n_cols;
    const uint32_t* beta_pows;  // device, 4 words per column
    const uint32_t* alpha;
    const uint32_t* tw;
    uint32_t* o0;
    uint32_t* o1;
    uint32_t* o2;
    uint32_t* o3;
    __device__ __forceinline__ SrcWideFold at(uint64_t) const { return *this; }
    // sum_c beta^c * v_c with 64-bit products accumulated unreduced: four
    // products fit on top of a folded accumulator (fold64), so accumulators are
    // folded after every group of four columns. A lifted
    // column gives the four f indices two values (rows r, r + 1, repeated), so
    // the lifted columns are summed first into two accumulators, which then
    // start the four of the full-size columns: 32 fewer registers than keeping
    // both sets, and no prefetched group, leave five waves a SIMD instead of
    // three (34 columns, 2^21 leaves: 219 -> 180 us).
    template <bool PRIO = true>
    __device__ __forceinline__ void pair(uint64_t i, uint32_t h[8]) const {
        const uint64_t j = 2 * i;  // f index of the first of four inputs (a multiple of 4)
        ConstLiftCol* tab = const_table(cols);
        ConstU32* bp = (ConstU32*)beta_pows;
        constexpr uint32_t G = 4;
        uint64_t ag[2][4] = {};
        uint32_t c = 0;
        while (c < n_cols && tab[c].sh != 0) {
            u32x2 v[G];
            uint32_t n = 0;  // lifted columns in this group
#pragma unroll
            for (uint32_t g = 0; g < G; g++) {
                v[g] = u32x2{0u, 0u};
                if (c + g < n_cols && tab[c + g].sh != 0) {
                    v[g] = *(GlobalV2*)(tab[c + g].p + ((j >> tab[c + g].sh) << 1));
                    n = g + 1;
                }
            }
#pragma unroll
            for (uint32_t g = 0; g < G; g++) {
                if (g >= n) break;
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const uint64_t w = bp[4 * (c + g) + m];
                    ag[0][m] += w * v[g].x;
                    ag[1][m] += w * v[g].y;
                }
            }
#pragma unroll
            for (int m = 0; m < 4; m++) {
                ag[0][m] = fold64(ag[0][m]);
                ag[1][m] = fold64(ag[1][m]);
            }
            c += n;
        }
        uint64_t af[4][4];
#pragma unroll
        for (int k = 0; k < 4; k++)
            for (int m = 0; m < 4; m++) af[k][m] = ag[k & 1][m];
        for (; c < n_cols; c += G) {
            u32x4 v[G];
#pragma unroll
            for (uint32_t g = 0; g < G; g++)
                if (c + g < n_cols) v[g] = *(GlobalV4*)(tab[c + g].p + j);
#pragma unroll
            for (uint32_t g = 0; g < G; g++) {
                if (c + g >= n_cols) break;
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const uint64_t w = bp[4 * (c + g) + m];
                    af[0][m] += w * v[g].x;
                    af[1][m] += w * v[g].y;
                    af[2][m] += w * v[g].z;
                    af[3][m] += w * v[g].w;
                }
            }
#pragma unroll
            for (int m = 0; m < 4; m++)
                for (int k = 0; k < 4; k++) af[k][m] = fold64(af[k][m]);
        }
        QM31 f[4];
#pragma unroll
        for (int k = 0; k < 4; k++)
            for (int m = 0; m < 4; m++) f[k].v[m] = reduce64(af[k][m]);
        const QMatrix al(load_alpha(alpha));
        const uint2 w = *(const uint2*)(tw + i);
        const QM31 g0 = fold_pair(f[0], f[1], al, w.x);
        const QM31 g1 = fold_pair(f[2], f[3], al, w.y);
        *(uint2*)(o0 + i) = make_uint2(g0.v[0], g1.v[0]);
        *(uint2*)(o1 + i) = make_uint2(g0.v[1], g1.v[1]);
        *(uint2*)(o2 + i) = make_uint2(g0.v[2], g1.v[2]);
        *(uint2*)(o3 + i) = make_uint2(g0.v[3], g1.v[3]);
        b2s_leaf_pair4<PRIO>(g0, g1, h);
    }
};

// ---------------------------------------------------------------- narrow levels
// Reduces n (a power of two <= 64) nodes stored node-major ([node][8 words]) in
// the LDS buffer `a` to `stop` nodes (a power of two) with the quads of the
// calling wave, ping-ponging with `b`. The buffers are 16-byte aligned. The nodes
// are at tree level `lvl`, node 0 having index idx0 there. Every lane of the
// wave must call this; returns the buffer holding the remaining nodes.
// A level is a lone wave's instruction count, so what does not change from
// level to level (and the level store's addresses) stays out of it.
__device__ __forceinline__ uint32_t* narrow_reduce(uint32_t* a, uint32_t* b, uint32_t n, uint32_t lvl, uint64_t idx0,
                                                   const LevelStore& st, uint32_t stop) {
    const uint32_t lane = threadIdx.x & 63, quad = lane >> 2, l = lane & 3;
    n = __builtin_amdgcn_readfirstlane(n);
    lvl = __builtin_amdgcn_readfirstlane(lvl);
    uint32_t h0, h1;
    b2s_quad_init(h0, h1);
    // this quad's place in the level store
    const bool store = st.base != nullptr;
    uint32_t* dst = store ? st.at(lvl + 1, idx0 >> 1) + 8 * quad + l : nullptr;
    while (n > stop) {
        const uint32_t half = n / 2;
        const bool want = store && lvl + 1 >= st.from && lvl + 1 <= st.depth;
        for (uint32_t q0 = 0; q0 < half; q0 += 16) {
            const uint32_t q = q0 + quad;
            const uint32_t qq = min(q, half - 1);  // whole quads stay active for the DPP permutes
            uint32_t hl = h0, hh = h1;
            b2s_compress_quad(a + 16 * qq, 64u, 0xFFFFFFFFu, hl, hh);
            if (q < half) {
                b[8 * q + l] = hl;
                b[8 * q + 4 + l] = hh;
                if (want) {
                    dst[8 * q0] = hl;
                    dst[8 * q0 + 4] = hh;
                }
            }
        }
        VX_WAVE_SYNC();
        lvl++;
        idx0 >>= 1;
        if (store) dst = st.at(lvl + 1, idx0 >> 1) + 8 * quad + l;
        uint32_t* t = a;
        a = b;
        b = t;
        n = half;
    }
    return a;
}

// The root of n (a power of two <= 64) such nodes: words l and 4 + l in rl, rh of
// lane l of every quad. The last level stays in registers, where the transcript
// hashes it. (Handing every level on in registers, a swap of lanes and sixteen
// DPP moves a level, takes 805 ns a level where this exchange takes 770: the moves
// stand before the rounds' chain, about 680 by itself, as the LDS trip does.)
__device__ __forceinline__ void narrow_root(uint32_t* a, uint32_t* b, uint32_t n, uint32_t lvl, uint64_t idx0,
                                            const LevelStore& st, uint32_t& rl, uint32_t& rh) {
    const uint32_t lane = threadIdx.x & 63, l = lane & 3;
    n = __builtin_amdgcn_readfirstlane(n);
    lvl = __builtin_amdgcn_readfirstlane(lvl);
    if (n == 1) {
        rl = a[l];
        rh = a[4 + l];
        return;
    }
    if (n > 2) {
        const uint32_t down = 30 - __builtin_clz(n);
        a = narrow_reduce(a, b, n, lvl, idx0, st, 2);
        lvl += down;
        idx0 >>= down;
    }
    b2s_quad_init(rl, rh);
    b2s_compress_quad(a, 64u, 0xFFFFFFFFu, rl, rh);
    if (st.want(lvl + 1) && lane < 4) {
        uint32_t* dst = st.at(lvl + 1, idx0 >> 1);
        dst[l] = rl;
        dst[4 + l] = rh;
    }
}

// One level of a block: the half = n / 2 parents (at most THREADS / 4, and a
// multiple of 16) of the nodes at `in` go to `out`, a quad per parent; the
// parents' level is lvl + 1, their first index idx0 >> 1.
__device__ __forceinline__ void block_quad_level(const uint32_t* in, uint32_t* out, uint32_t half, uint32_t lvl,
                                                 uint64_t idx0, const LevelStore& st) {
    const uint32_t quad = threadIdx.x >> 2, l = threadIdx.x & 3;
    if ((threadIdx.x >> 6) * 16 < half) {  // wave-uniform
        uint32_t hl, hh;
        b2s_quad_init(hl, hh);
        b2s_compress_quad(in + 16 * quad, 64u, 0xFFFFFFFFu, hl, hh);
        out[8 * quad + l] = hl;
        out[8 * quad + 4 + l] = hh;
        if (st.want(lvl + 1)) {
            uint32_t* dst = st.at(lvl + 1, (idx0 >> 1) + quad);
            dst[l] = hl;
            dst[4 + l] = hh;
        }
    }
}
// n nodes (a power of two) node-major in the LDS buffer a down to at most 32,
// ping-ponging with b: a level costs one quad compression of latency while its
// waves have a SIMD each. All threads of the block must call it, the buffer
// complete; afterwards a holds the remaining nodes.
__device__ __forceinline__ void block_quad_reduce(uint32_t*& a, uint32_t*& b, uint32_t& n, uint32_t& lvl,
                                                  uint64_t& idx0, const LevelStore& st) {
    while (n > 32) {
        block_quad_level(a, b, n / 2, lvl, idx0, st);
        lds_barrier();
        uint32_t* t = a;
        a = b;
        b = t;
        n /= 2;
        lvl++;
        idx0 >>= 1;
    }
}

// The transcript while a wave holds it, in registers: lane l of every quad has
// state words l and 4 + l (channel.rs:15-25).
struct QuadTranscript {
    uint32_t sl, sh, n_draws, failed;
    __device__ __forceinline__ void load(const DevChannel* ch, bool init) {
        const uint32_t l = threadIdx.x & 3;
        sl = init ? 0u : ch->state[l];
        sh = init ? 0u : ch->state[4 + l];
        failed = init ? 0u : ch->failed;
        n_draws = 0;
    }
    // H(state || second half) with t bytes counted
    __device__ __forceinline__ void hash(uint32_t xl, uint32_t xh, uint32_t t, uint32_t& hl, uint32_t& hh) const {
        uint32_t m[16];
        quad_gather(sl, m);
        quad_gather(sh, m + 4);
        quad_gather(xl, m + 8);
        quad_gather(xh, m + 12);
        b2s_quad_init(hl, hh);
        b2s_compress_quad_words(m, t, 0xFFFFFFFFu, hl, hh);
    }
    // mix_digest (channel.rs:30-39) of the root words of lane l
    __device__ __forceinline__ void mix(uint32_t rl, uint32_t rh) {
        uint32_t nl, nh;
        hash(rl, rh, 64u, nl, nh);
        sl = nl;
        sh = nh;
        n_draws = 0;
    }
    // draw_felt (channel.rs:67-86); lane l gets word l. False when the retry
    // budget is exhausted.
    __device__ __forceinline__ bool draw(uint32_t& w) {
        const uint32_t l = threadIdx.x & 3;
        for (int tries = 0; tries < 64; tries++) {
            uint32_t wl, wh;
            hash(l == 0 ? n_draws : 0u, 0u, 37u, wl, wh);
            n_draws++;
            const uint64_t ok = __ballot(wl < 2u * P && wh < 2u * P);
            if ((ok & 0xFull) == 0xFull) {
                w = canon(wl);
                return true;
            }
        }
        failed = 1;
        return false;
    }
    __device__ __forceinline__ void store(DevChannel* ch) const {
        const uint32_t lane = threadIdx.x & 63, l = lane & 3;
        if (lane < 4) {
            ch->state[l] = sl;
            ch->state[4 + l] = sh;
        }
        if (lane == 0) {
            ch->n_draws = n_draws;
            ch->failed = failed;
        }
    }
};

// ---------------------------------------------------------------- stage kernel
// A source may cap logc_max (STAGE_LOGC_MAX): leaves that take more work each
// fill the device at a smaller depth.
template <class S, class = void>
struct StageLogcMax {
    static constexpr uint32_t value = MERKLE_LOGC_MAX;
};
template <class S>
struct StageLogcMax<S, std::void_t<decltype(S::STAGE_LOGC_MAX)>> {
    static constexpr uint32_t value = S::STAGE_LOGC_MAX;
};
// The tuned depth table is timed on single-column leaves; a source that caps
// its depth takes the default rule of pick_stage instead.
template <class S>
constexpr bool stage_uses_plan() {
    return StageLogcMax<S>::value == MERKLE_LOGC_MAX;
}
// LDS words of a stage wave: one slot of 64 nodes per pending level of its
// binary counter, and room for the 64 -> keep reduction (64 nodes and the next
// level's 32).
__host__ __device__ inline uint32_t stage_wave_words(uint32_t logc) { return logc >= 2 ? logc * 512 : 768; }
inline uint32_t stage_lds_bytes(uint32_t logc) { return 4 * MERKLE_STAGE_WAVES * stage_wave_words(logc); }

// blockIdx.y selects the proof of a batch: every per-proof buffer (items,
// out_nodes, level store) lies blockIdx.y * bs words past proof 0's.
// A wave hands on `keep` (a power of two <= 32) nodes of its subtree: the last
// levels of its 64 -> 1 reduction leave most of the wave's quads idle, and the
// next stage computes those nodes one per lane instead. Dynamic LDS:
// stage_lds_bytes(logc).
template <class Src>
__global__ __launch_bounds__(64 * MERKLE_STAGE_WAVES) void merkle_stage_kernel(Src src0, uint32_t item_level,
                                                                             uint64_t n_items, uint32_t logc,
                                                                             uint32_t* out_nodes, LevelStore st0,
                                                                             uint64_t bs, uint32_t keep) {
    extern __shared__ __align__(16) uint32_t stage_lds[];
    const uint64_t boff = (uint64_t)blockIdx.y * bs;
    const Src src = src0.at(boff);
    const LevelStore st = st0.shifted(boff);
    out_nodes += boff;
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t* wl = stage_lds + w * stage_wave_words(logc);
    const uint64_t wave_id = (uint64_t)blockIdx.x * MERKLE_STAGE_WAVES + w;
    const uint64_t base = wave_id << (7 + logc);
    if (base >= n_items) return;  // wave-uniform
    const uint32_t n_chunks = 1u << logc;
    uint32_t h[8];
    for (uint32_t c = 0; c < n_chunks; c++) {
        const uint64_t i = base + 128ull * c + 2 * lane;
        src.pair(i, h);
        uint32_t lvl = item_level + 1, d = 0, k = c;
        if (st.want(lvl)) store8(st.at(lvl, i >> 1), h);
        while (k & 1) {
            // The left sibling chunk waits in slot d, the right chunk is h: lanes
            // 0-31 take the left chunk's pairs, then h takes the slot and lanes
            // 32-63 its pairs. Slots hold 64 nodes word-major ([word][lane]).
            uint32_t* slot = wl + d * 512;
            const uint32_t li = (lane & 31) * 2;
            uint32_t l[8], r[8];
            if (lane < 32) {
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    l[q] = slot[q * 64 + li];
                    r[q] = slot[q * 64 + li + 1];
                }
            }
            VX_WAVE_SYNC();
#pragma unroll
            for (int q = 0; q < 8; q++) slot[q * 64 + lane] = h[q];
            VX_WAVE_SYNC();
            if (lane >= 32) {
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    l[q] = slot[q * 64 + li];
                    r[q] = slot[q * 64 + li + 1];
                }
            }
            VX_WAVE_SYNC();
            b2s_node(l, r, h);
            lvl++;
            d++;
            k >>= 1;
            if (st.want(lvl)) {
                uint64_t idx = (base >> (lvl - item_level)) + 64ull * (c >> d) + lane;
                store8(st.at(lvl, idx), h);
            }
        }
        if (c + 1 < n_chunks) {
#pragma unroll
            for (int q = 0; q < 8; q++) wl[d * 512 + q * 64 + lane] = h[q];
            VX_WAVE_SYNC();
        }
    }
    // the wave's 64 top nodes (level item_level + 1 + logc) -> `keep` nodes
#pragma unroll
    for (int q = 0; q < 8; q++) wl[lane * 8 + q] = h[q];
    VX_WAVE_SYNC();
    const uint32_t* top = narrow_reduce(wl, wl + 512, 64, item_level + 1 + logc, wave_id * 64, st, keep);
    for (uint32_t k = lane; k < 8 * keep; k += 64) out_nodes[8 * keep * wave_id + k] = top[k];
}

// ---------------------------------------------------------------- small leaf stages
// Leaf stage of a small tree: one leaf per quad, hashed quad-cooperatively,
// 16 * R leaves a wave reduced to one node, a workgroup's four to one. On the few
// waves such a tree has (at most one per SIMD), a wave's chain is then R quad
// compressions for the leaves and log2(64 R) node levels, where the lane-per-pair
// form (128 leaves a wave) takes three lane compressions and seven quad rounds. The
// last two levels cost two quad compressions of one wave and save the tail kernel
// its two widest levels, which are its dearest (three more, of eight waves a
// workgroup, cost more than they save). Every lane of a quad forms its leaf's words.
constexpr uint32_t LEAF_QUAD_WAVES = 4;  // waves per workgroup
template <class Src, uint32_t R>
__global__ __launch_bounds__(64 * LEAF_QUAD_WAVES) void leaf_quad_stage_kernel(Src src0, uint32_t* out_nodes,
                                                                             LevelStore st0, uint64_t bs) {
    constexpr uint32_t LPW = 16 * R;  // leaves a wave
    __shared__ __align__(16) uint32_t lds[LEAF_QUAD_WAVES][8 * LPW + 4 * LPW];
    __shared__ __align__(16) uint32_t tops[8 * LEAF_QUAD_WAVES], tops2[4 * LEAF_QUAD_WAVES];
    const uint64_t boff = (uint64_t)blockIdx.y * bs;
    const Src src = src0.at(boff);
    const LevelStore st = st0.shifted(boff);
    out_nodes += boff;
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6, quad = lane >> 2, l = lane & 3;
    const uint64_t wave_id = (uint64_t)blockIdx.x * LEAF_QUAD_WAVES + w;
    const uint64_t base = wave_id * LPW;  // n_items is a multiple of the block's leaves
    uint32_t* na = lds[w];                // LPW nodes, node-major
    uint32_t* nb = na + 8 * LPW;          // the next level
    for (uint32_t r = 0; r < R; r++) {
        const uint32_t k = 16 * r + quad;
        uint32_t v[Src::WIDTH], hl, hh;
        src.words(base + k, l, v);
        b2s_leaf_quad<Src::WIDTH>(v, hl, hh);
        na[8 * k + l] = hl;
        na[8 * k + 4 + l] = hh;
    }
    VX_WAVE_SYNC();
    uint32_t rl, rh;
    narrow_root(na, nb, LPW, 0, base, st, rl, rh);
    if (lane < 4) {
        tops[8 * w + lane] = rl;
        tops[8 * w + 4 + lane] = rh;
    }
    lds_barrier();
    if (w) return;
    constexpr uint32_t LOG = R == 1 ? 4 : R == 2 ? 5 : 6;
    narrow_root(tops, tops2, LEAF_QUAD_WAVES, LOG, (uint64_t)blockIdx.x * LEAF_QUAD_WAVES, st, rl, rh);
    if (lane < 4) {
        out_nodes[8ull * blockIdx.x + lane] = rl;
        out_nodes[8ull * blockIdx.x + 4 + lane] = rh;
    }
}

// ---------------------------------------------------------------- tail kernel
struct TailOut {
    uint32_t* root_dst;      // 8 words (e.g. inside the proof buffer); may be null
    DevChannel* channel;     // transcript to advance; may be null
    uint32_t* alpha_dst;     // challenges drawn after mixing the root; may be null
    uint32_t init_channel;   // reset the transcript before mixing
    uint32_t n_felts = 1;    // challenges drawn (4 words each)
};

constexpr uint32_t TAIL_THREADS = 1024;
// Most nodes of a level whose parents are hashed by quads: 128 parents are eight
// waves, two a SIMD (measured against one parent a lane at the same width, the
// quads of 128 parents are faster, of 256 slower).
constexpr uint32_t TAIL_QUAD_NODES = 256;

template <class S>
struct IsNodes : std::false_type {};
template <>
struct IsNodes<SrcNodes> : std::true_type {};

// Lane-per-parent levels of a block: m nodes word-major in `nodes` (word q of
// node j at q * W + j) down to TAIL_QUAD_NODES nodes, which end node-major in
// out; the caller synchronises before. The nodes are at level lvl.
template <uint32_t W>
__device__ __forceinline__ void block_lane_levels(uint32_t* nodes, uint32_t* out, uint32_t& m, uint32_t& lvl,
                                                  uint64_t idx0, const LevelStore& st) {
    const uint32_t tid = threadIdx.x;
    while (m > TAIL_QUAD_NODES) {
        const uint32_t half = m / 2;
        uint32_t l[8], r[8];
        if (tid < half) {
#pragma unroll
            for (int q = 0; q < 8; q++) {
                l[q] = nodes[q * W + 2 * tid];
                r[q] = nodes[q * W + 2 * tid + 1];
            }
        }
        lds_barrier();
        lvl++;
        idx0 >>= 1;
        if (tid < half) {
            uint32_t h[8];
            if (half > TAIL_QUAD_NODES) {
                b2s_node(l, r, h);
#pragma unroll
                for (int q = 0; q < 8; q++) nodes[q * W + tid] = h[q];
            } else {
                b2s_node<false>(l, r, h);  // one wave a SIMD
                store8(out + 8 * tid, h);
            }
            if (st.want(lvl)) store8(st.at(lvl, idx0 + tid), h);
        }
        lds_barrier();
        m = half;
    }
}

// Block b reduces items [b * n_items, (b + 1) * n_items) to one root (the
// tiled form used by the reference-ABI entry points runs many blocks; the
// prover runs one). n_items is a power of two in [2, MERKLE_TAIL_MAX].
// blockIdx.y selects the proof of a batch as in merkle_stage_kernel; the root,
// transcript and challenge destinations move with it.
//
// A chain of dependent levels: one lane compression (about 1.7 us) a level
// while it has more than 128 parents, one quad compression (0.76 us with its exchange) below,
// then the transcript's two. The transcript's state is fetched before the first
// level, and the last level writes the root where the transcript hashes it.
// PRIO = false: the first level's waves have a SIMD each; FEW: at most 16 nodes
// (launch_tail).
template <class Src, bool PRIO, bool FEW>
__global__ __launch_bounds__(TAIL_THREADS) void merkle_tail_kernel(Src src0, uint32_t item_level, uint32_t n_items,
                                                                  LevelStore st0, TailOut out, uint64_t bs) {
    constexpr uint32_t W = MERKLE_TAIL_MAX / 2;
    const uint64_t boff = (uint64_t)blockIdx.y * bs;
    const Src src = src0.at(boff);
    const LevelStore st = st0.shifted(boff);
    if (boff) {
        if (out.root_dst) out.root_dst += boff;
        if (out.channel) out.channel = (DevChannel*)((uint32_t*)out.channel + boff);
        if (out.alpha_dst) out.alpha_dst += boff;
    }
    __shared__ uint32_t nodes[8 * W];
    __shared__ __align__(16) uint32_t qa[8 * TAIL_QUAD_NODES], qb[4 * TAIL_QUAD_NODES];
    const uint32_t tid = threadIdx.x;
    const uint64_t item_base = (uint64_t)blockIdx.x * n_items;
    QuadTranscript tr = {};
    if (out.channel && tid < 64) tr.load(out.channel, out.init_channel != 0);
    uint32_t n = n_items / 2, lvl = item_level + 1;
    bool narrow = false;
    if constexpr (IsNodes<Src>::value) narrow = FEW || (n_items <= TAIL_QUAD_NODES && n_items > 16);
    if (narrow) {
        if constexpr (IsNodes<Src>::value && FEW) {  // all levels by one wave
            if (tid < 8 * n_items) qa[tid] = src.nodes[8 * item_base + tid];
            n = n_items;
            lvl = item_level;
        } else if constexpr (IsNodes<Src>::value) {
            // the first level's quads read the nodes in place
            block_quad_level(src.nodes + 8 * item_base, qa, n, item_level, item_base, st);
        }
        lds_barrier();
    } else {
        for (uint32_t j = tid; j < n; j += TAIL_THREADS) {
            uint32_t h[8];
            src.template pair<PRIO>(item_base + 2ull * j, h);
            if (st.want(lvl)) store8(st.at(lvl, (item_base >> 1) + j), h);
            if (n > TAIL_QUAD_NODES) {
#pragma unroll
                for (int q = 0; q < 8; q++) nodes[q * W + j] = h[q];
            } else {
                store8(qa + 8 * j, h);
            }
        }
        lds_barrier();
        block_lane_levels<W>(nodes, qa, n, lvl, item_base >> (lvl - item_level), st);
    }
    uint64_t idx0 = item_base >> (lvl - item_level);
    uint32_t *cur = qa, *nxt = qb;
    block_quad_reduce(cur, nxt, n, lvl, idx0, st);
    if (tid >= 64) return;  // one wave finishes: narrow levels and transcript
    uint32_t rl, rh;
    narrow_root(cur, nxt, n, lvl, idx0, st, rl, rh);
    if (out.root_dst && tid < 4) {
        out.root_dst[8ull * blockIdx.x + tid] = rl;
        out.root_dst[8ull * blockIdx.x + 4 + tid] = rh;
    }
    if (!out.channel) return;
    tr.mix(rl, rh);
    for (uint32_t k = 0; out.alpha_dst && k < out.n_felts; k++) {
        uint32_t w = 0;
        if (!tr.draw(w)) break;
        if (tid < 4) out.alpha_dst[4 * k + tid] = w;
    }
    tr.store(out.channel);
}

// Tail of `batch` proofs (one block each, all at once on the device up to 256).
// A first level of at most 256 parents is one wave a SIMD of its block's CU, which
// hashes without priorities (roots of 2 and 16 leaves: 7.8 and 10.25 us with them, 7.25
// and 9.85 without).
template <class Src>
inline void launch_tail(const Src& src, uint32_t item_level, uint32_t n_items, LevelStore st, TailOut out, uint32_t batch,
                        uint64_t bs, hipStream_t s) {
    const dim3 grid(1, batch);
    if constexpr (IsNodes<Src>::value) {
        // nodes that one wave's quads can hash from the first level on; a kernel of its
        // own, since the choice costs the one for more nodes 0.5 us
        if (n_items <= 16) {
            merkle_tail_kernel<Src, false, true><<<grid, TAIL_THREADS, 0, s>>>(src, item_level, n_items, st, out, bs);
            return;
        }
    }
    if (n_items <= 512 && batch <= LONE_THREADS / 256)
        merkle_tail_kernel<Src, false, false><<<grid, TAIL_THREADS, 0, s>>>(src, item_level, n_items, st, out, bs);
    else
        merkle_tail_kernel<Src, true, false><<<grid, TAIL_THREADS, 0, s>>>(src, item_level, n_items, st, out, bs);
}

}  // namespace vx
