// Reference-ABI Blake2s Merkle entry points (cuda/blake2s.cu:522-632) on top of
// the wave64 engine. Hash values and tree shapes are the reference's; the
// tiled forms return the root of every 1024-leaf tile.
#include "common.hpp"
#include "merkle_engine.hpp"

namespace vx {

// Up to 16 columns behind a device pointer array; leaf uses the first
// min(n_cols, 16) columns and t = 4 * min(n_cols, 16) (cuda/blake2s.cu:25-60).
// NC > 0: exactly NC columns, whose zero message words are known at compile
// time (one column is the trace's, four a QM31 column's); NC = 0: any number.
template <uint32_t NC>
struct SrcCols {
    const uint32_t* const* cols;
    uint32_t n_cols;
    __device__ __forceinline__ SrcCols at(uint64_t) const { return *this; }
    // the words of K consecutive leaves from i on
    template <uint32_t K, bool PRIO = true>
    __device__ __forceinline__ void hash(uint64_t i, uint32_t h[K][8]) const {
        if constexpr (NC > 0) {
            uint32_t w[K][NC];
#pragma unroll
            for (uint32_t c = 0; c < NC; c++) {
                const gu32* p = as_global(cols[c]);
#pragma unroll
                for (uint32_t k = 0; k < K; k++) w[k][c] = p[i + k];
            }
            b2s_leaves<K, NC, PRIO>(w, h);
        } else {
            const uint32_t eff = n_cols > 16 ? 16 : n_cols;
            uint32_t m[K][16];
#pragma unroll
            for (uint32_t c = 0; c < 16; c++) {
#pragma unroll
                for (uint32_t k = 0; k < K; k++) m[k][c] = c < eff ? as_global(cols[c])[i + k] : 0u;
            }
#pragma unroll
            for (uint32_t k = 0; k < K; k++) b2s_init(h[k]);
            b2s_compress_n<K, 16, PRIO>(h, m, 4u * eff, 0xFFFFFFFFu);
        }
    }
    template <bool PRIO = true>
    __device__ __forceinline__ void pair(uint64_t i, uint32_t h[8]) const {
        uint32_t l[2][8];
        hash<2, PRIO>(i, l);
        b2s_node<PRIO>(l[0], l[1], h);
    }
};

// A leaf a lane; PRIO = false for launches whose waves have a SIMD each (us at
// 2^15 leaves of 16 columns: 4.35 with priorities, 4.10 without).
template <uint32_t NC, bool PRIO>
__global__ __launch_bounds__(256) void hash_leaves_kernel(SrcCols<NC> src, uint32_t* out, uint32_t n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    uint32_t h[1][8];
    src.template hash<1, PRIO>(i, h);
    store8(out + 8ull * i, h[0]);
}

// Root of every tile of TILE_LEAVES leaves. Bound by the chain of one tile while
// there are few, by the hashing when there are many (us for one column, before:
// the tail kernel of 1024 threads a tile):
// - FEW, one workgroup of 1024 threads a tile: a pair of leaves a lane of the
//   first eight waves, the 512 nodes then down by quads, 256 of them on the first
//   level: three lane and nine quad compressions. 16 tiles: 23 -> 17.4.
// - otherwise 256 threads a tile: a wave hashes its 256 leaves as two chunks and
//   merges them as merkle_stage_kernel does; a level by lanes, then quads: eight
//   lane and seven quad compressions, but no lane idle in the first five.
//   1024 tiles (the hashing takes 30 at full rate): 67 -> 46, FEW 53.
// - from TILE_STAGE_MIN tiles on a wave a tile keeps every SIMD full by itself
//   and wastes no lane on the middle levels: merkle_stage_kernel at depth 3, whose
//   wave covers exactly 1024 leaves. 16384 tiles: 543 -> 513, 4096: 143 -> 142.
constexpr uint32_t TILE_LEAVES = 1024;
constexpr uint32_t TILE_FEW_MAX = 256;
constexpr uint32_t TILE_STAGE_MIN = 4096;
template <class Src, bool FEW>
__global__ __launch_bounds__(FEW ? 1024 : 256) void merkle_tile_kernel(Src src, uint32_t* roots) {
    __shared__ __align__(16) uint32_t na[FEW ? 8 * 512 : 8 * 256], nb[FEW ? 8 * 256 : 8 * 128];
    const LevelStore none = {nullptr, 0, 0};
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    uint32_t h[8];
    uint32_t *cur, *nxt, n, lvl = 0;
    uint64_t idx0 = 0;
    if constexpr (FEW) {
        if (tid < 512) {
            src.pair((uint64_t)blockIdx.x * TILE_LEAVES + 2 * tid, h);
            store8(na + 8 * tid, h);
        }
        lds_barrier();
        cur = na;
        nxt = nb;
        n = 512;
    } else {
        const uint64_t base = (uint64_t)blockIdx.x * TILE_LEAVES + 256 * (tid >> 6);
        uint32_t* slot = na + 512 * (tid >> 6);  // the wave's first chunk, then its 64 nodes
        uint32_t l[8], r[8];
        src.pair(base + 2 * lane, h);
#pragma unroll
        for (int q = 0; q < 8; q++) slot[q * 64 + lane] = h[q];
        src.pair(base + 128 + 2 * lane, h);
        const uint32_t li = (lane & 31) * 2;
        VX_WAVE_SYNC();
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
        store8(slot + 8 * lane, h);
        lds_barrier();
        if (tid < 128) {
            load8(na + 16 * tid, l);
            load8(na + 16 * tid + 8, r);
            b2s_node(l, r, h);
            store8(nb + 8 * tid, h);
        }
        lds_barrier();
        cur = nb;
        nxt = na;
        n = 128;
    }
    block_quad_reduce(cur, nxt, n, lvl, idx0, none);
    if (tid >= 64) return;
    uint32_t rl, rh;
    narrow_root(cur, nxt, n, lvl, idx0, none, rl, rh);
    if (tid < 4) {
        roots[8ull * blockIdx.x + tid] = rl;
        roots[8ull * blockIdx.x + 4 + tid] = rh;
    }
}

// A level of a tree, one parent a lane. While the launch has at most one wave a
// SIMD the compression goes without priorities, which a lone wave only waits for;
// up to NODES_QUAD_MAX parents a quad each, a shorter chain (3.4 us a small
// level with priorities, 1.8 by quads).
constexpr uint32_t NODES_QUAD_MAX = 1u << 14;
template <bool PRIO>
__global__ __launch_bounds__(256) void hash_nodes_kernel(const uint32_t* ch, uint32_t* par, uint32_t n) {
    uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    uint32_t l[8], r[8], h[8];
    load8(ch + 16ull * i, l);
    load8(ch + 16ull * i + 8, r);
    b2s_node<PRIO>(l, r, h);
    store8(par + 8ull * i, h);
}
__global__ __launch_bounds__(256) void hash_nodes_quad_kernel(const uint32_t* ch, uint32_t* par, uint32_t n) {
    const uint32_t i = blockIdx.x * 64 + (threadIdx.x >> 2), l = threadIdx.x & 3;
    uint32_t hl, hh;
    b2s_quad_init(hl, hh);
    b2s_compress_quad(ch + 16ull * min(i, n - 1), 64u, 0xFFFFFFFFu, hl, hh);  // whole quads stay active
    if (i >= n) return;
    par[8ull * i + l] = hl;
    par[8ull * i + 4 + l] = hh;
}
// A pair of leaves and their parent a lane (2^13 leaves: 7.3 us with priorities, 6.6 without).
template <bool PRIO>
__global__ void leaves_merge_soa4_kernel(SrcSoa4 src, uint32_t* par, uint32_t n_pairs) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_pairs) return;
    uint32_t h[8];
    src.pair<PRIO>(2ull * i, h);
    store8(par + 8ull * i, h);
}
__global__ void copy8_kernel(const uint32_t* s, uint32_t* d) {
    if (threadIdx.x < 8) d[threadIdx.x] = s[threadIdx.x];
}

template <uint32_t NC>
static void hash_leaves(SrcCols<NC> src, uint32_t* hashes, uint32_t n) {
    const uint32_t grid = ceil_div(n, 256);
    if (n <= LONE_THREADS)
        hash_leaves_kernel<NC, false><<<grid, 256, 0, current_stream()>>>(src, hashes, n);
    else
        hash_leaves_kernel<NC, true><<<grid, 256, 0, current_stream()>>>(src, hashes, n);
}

template <class Src>
static void tail_root(Src src, uint32_t n_items, uint32_t* root, hipStream_t st, const char* what) {
    LevelStore none = {nullptr, 0, 0};
    TailOut out = {root, nullptr, nullptr, 0};
    launch_tail(src, 0, n_items, none, out, 1, 0, st);
    check_launch(what);
}

template <class Src>
static void tile_roots(Src src, uint32_t n_leaves, uint32_t* roots, hipStream_t st, const char* what) {
    const uint32_t tiles = n_leaves / TILE_LEAVES;
    if (!tiles) return;
    if (tiles >= TILE_STAGE_MIN) {
        const LevelStore none = {nullptr, 0, 0};
        merkle_stage_kernel<Src><<<ceil_div(tiles, MERKLE_STAGE_WAVES), 64 * MERKLE_STAGE_WAVES, stage_lds_bytes(3), st>>>(
            src, 0, (uint64_t)tiles * TILE_LEAVES, 3, roots, none, 0, 1u);
    } else if (tiles > TILE_FEW_MAX) {
        merkle_tile_kernel<Src, false><<<tiles, 256, 0, st>>>(src, roots);
    } else {
        merkle_tile_kernel<Src, true><<<tiles, 1024, 0, st>>>(src, roots);
    }
    check_launch(what);
}

}  // namespace vx

using namespace vx;

extern "C" {

void cuda_merkle_hash_leaves(const uint32_t* const* columns, uint32_t* hashes, uint32_t n_cols, uint32_t n_leaves) {
    if (!n_leaves) return;
    if (n_cols == 1)
        hash_leaves(SrcCols<1>{columns, n_cols}, hashes, n_leaves);
    else if (n_cols == 4)
        hash_leaves(SrcCols<4>{columns, n_cols}, hashes, n_leaves);
    else
        hash_leaves(SrcCols<0>{columns, n_cols}, hashes, n_leaves);
    check_launch("cuda_merkle_hash_leaves");
}

void cuda_merkle_hash_nodes(const uint32_t* children, uint32_t* parents, uint32_t n_parents) {
    if (!n_parents) return;
    if (n_parents <= NODES_QUAD_MAX)
        hash_nodes_quad_kernel<<<ceil_div(n_parents, 64), 256, 0, current_stream()>>>(children, parents, n_parents);
    else if (n_parents <= LONE_THREADS)
        hash_nodes_kernel<false><<<ceil_div(n_parents, 256), 256, 0, current_stream()>>>(children, parents, n_parents);
    else
        hash_nodes_kernel<true><<<ceil_div(n_parents, 256), 256, 0, current_stream()>>>(children, parents, n_parents);
    check_launch("cuda_merkle_hash_nodes");
}

void cuda_merkle_reduce_to_root(const uint32_t* nodes, uint32_t* root_out, uint32_t n_nodes) {
    if (n_nodes == 0) return;
    if (n_nodes == 1) {
        copy8_kernel<<<1, 64, 0, current_stream()>>>(nodes, root_out);
        check_launch("cuda_merkle_reduce_to_root");
        return;
    }
    if (!is_pow2(n_nodes) || n_nodes > MERKLE_TAIL_MAX) {
        set_error(-2, "cuda_merkle_reduce_to_root: n_nodes must be a power of two <= 4096");
        return;
    }
    tail_root(SrcNodes{nodes}, n_nodes, root_out, current_stream(), "cuda_merkle_reduce_to_root");
}

void cuda_merkle_commit_small_soa4(const uint32_t* c0, const uint32_t* c1, const uint32_t* c2, const uint32_t* c3,
                                   uint32_t* root_out, uint32_t n_leaves) {
    if (n_leaves < 2 || !is_pow2(n_leaves) || n_leaves > MERKLE_TAIL_MAX) {
        set_error(-2, "cuda_merkle_commit_small_soa4: n_leaves must be a power of two in [2, 4096]");
        return;
    }
    tail_root(SrcSoa4{c0, c1, c2, c3}, n_leaves, root_out, current_stream(), "cuda_merkle_commit_small_soa4");
}

void cuda_merkle_hash_leaves_merge_soa4(const uint32_t* c0, const uint32_t* c1, const uint32_t* c2,
                                        const uint32_t* c3, uint32_t* parents, uint32_t n_leaves) {
    uint32_t n_pairs = n_leaves / 2;
    if (!n_pairs) return;
    const SrcSoa4 src = {c0, c1, c2, c3};
    const uint32_t grid = ceil_div(n_pairs, 256);
    if (n_pairs <= LONE_THREADS)
        leaves_merge_soa4_kernel<false><<<grid, 256, 0, current_stream()>>>(src, parents, n_pairs);
    else
        leaves_merge_soa4_kernel<true><<<grid, 256, 0, current_stream()>>>(src, parents, n_pairs);
    check_launch("cuda_merkle_hash_leaves_merge_soa4");
}

void cuda_merkle_tiled_soa4(const uint32_t* c0, const uint32_t* c1, const uint32_t* c2, const uint32_t* c3,
                            uint32_t* subtree_roots, uint32_t n_leaves) {
    cuda_merkle_tiled_soa4_stream(c0, c1, c2, c3, subtree_roots, n_leaves, current_stream());
}

void cuda_merkle_tiled_soa4_stream(const uint32_t* c0, const uint32_t* c1, const uint32_t* c2, const uint32_t* c3,
                                   uint32_t* subtree_roots, uint32_t n_leaves, void* stream) {
    tile_roots(SrcSoa4{c0, c1, c2, c3}, n_leaves, subtree_roots, (hipStream_t)stream, "cuda_merkle_tiled_soa4");
}

void cuda_merkle_tiled_generic(const uint32_t* const* columns, uint32_t* subtree_roots, uint32_t n_cols,
                               uint32_t n_leaves) {
    const char* what = "cuda_merkle_tiled_generic";
    if (n_cols == 1)
        tile_roots(SrcCols<1>{columns, n_cols}, n_leaves, subtree_roots, current_stream(), what);
    else if (n_cols == 4)
        tile_roots(SrcCols<4>{columns, n_cols}, n_leaves, subtree_roots, current_stream(), what);
    else
        tile_roots(SrcCols<0>{columns, n_cols}, n_leaves, subtree_roots, current_stream(), what);
}

}  // extern "C"
