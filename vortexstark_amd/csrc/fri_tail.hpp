// The small FRI layers of a proof in one launch.
//
// Up to 1024 values a layer's fold, leaf hashes, tree and transcript step fit
// one workgroup, and launching kernels per layer costs more than the layer
// itself. fri_tail_kernel runs every remaining line fold of a proof in one
// workgroup of 1024 threads: fold (cuda/fri.cu:10-39) into the next layer,
// hash it as an SoA4 tree (level-store nodes written as by the stage/tail
// kernels), reduce to the root, mix the root into the transcript and draw the
// next challenge. A layer is a chain of about log2(n) + 3 dependent
// compressions, so what counts is the latency between them: a layer's values
// stay in LDS for the next fold, the next twiddles are fetched while a layer
// is hashed, and the transcript's state stays in the registers of one wave
// (device memory gets all of them, but nothing is read back from it). Leaves
// of layers of at most 128 values are hashed a quad each (0.7 us for up to
// 64), larger ones a lane each (1.7 us at one wave a SIMD). A 2048-value layer
// is left to a stage launch and a tree tail: its 4095 compressions in one
// workgroup are bound by one CU's issue rate.
// blockIdx.y selects the proof of a batch (buffers bs words apart).
#pragma once
#include "merkle_engine.hpp"

namespace vx {

constexpr uint32_t FRI_TAIL_MAX_LAYERS = 12;
constexpr uint32_t FRI_TAIL_MAX_ITEMS = 1024;  // values of the largest layer handled here
constexpr uint32_t FRI_TAIL_THREADS = 1024;
static_assert(FRI_TAIL_MAX_ITEMS <= FRI_TAIL_THREADS, "one leaf per thread");

struct FriTailLayer {
    const uint32_t* in[4];   // previous layer, 2n values per column
    uint32_t* out[4];        // this layer, n values per column
    const uint32_t* tw;      // n fold twiddles (shared by a batch)
    uint32_t* root_dst;      // 8 words
    uint32_t* alpha_dst;     // next layer's challenge (null after the last layer)
    LevelStore st;
    uint32_t n;              // values of this layer: a power of two in [2, FRI_TAIL_MAX_ITEMS]
};
struct FriTailArgs {
    FriTailLayer L[FRI_TAIL_MAX_LAYERS];
    uint32_t n_layers;
    const uint32_t* alpha0;  // challenge of the first layer
    DevChannel* channel;
};

constexpr uint32_t FRI_TAIL_QUAD_LEAVES = 128;  // largest layer whose leaves are hashed by quads

static __global__ __launch_bounds__(FRI_TAIL_THREADS) void fri_tail_kernel(FriTailArgs args, uint64_t bs) {
    constexpr uint32_t W = FRI_TAIL_MAX_ITEMS;
    __shared__ uint32_t nodes[8 * W];  // wide levels, word-major
    __shared__ __align__(16) uint32_t qa[8 * TAIL_QUAD_NODES], qb[4 * TAIL_QUAD_NODES];
    __shared__ __align__(8) uint32_t val[4][W];  // the layer's values
    __shared__ uint32_t al[4];
    const uint32_t tid = threadIdx.x;
    const uint64_t boff = (uint64_t)blockIdx.y * bs;
    DevChannel* ch = (DevChannel*)((uint32_t*)args.channel + boff);
    QuadTranscript tr = {};
    if (tid < 64) {
        tr.load(ch, false);
        if (tid < 4) al[tid] = args.alpha0[boff + tid];
    }
    // value index of this thread in a layer of n values: a quad per value in the
    // layers whose leaves quads hash
    auto slot = [&](uint32_t n) { return n <= FRI_TAIL_QUAD_LEAVES ? tid >> 2 : tid; };
    uint32_t n = args.L[0].n;
    uint32_t k = slot(n);
    uint2 in[4];
    uint32_t tw = 0;
    if (k < n) {
        tw = args.L[0].tw[k];
#pragma unroll
        for (int c = 0; c < 4; c++) in[c] = *(const uint2*)(args.L[0].in[c] + boff + 2 * k);
    }
    lds_barrier();
    for (uint32_t li = 0; li < args.n_layers; li++) {
        const FriTailLayer& L = args.L[li];
        const LevelStore st = L.st.shifted(boff);
        const bool quads = n <= FRI_TAIL_QUAD_LEAVES;
        const bool more = li + 1 < args.n_layers;
        const uint32_t k1 = slot(n / 2);
        uint32_t tw1 = 0;
        if (more && k1 < n / 2) tw1 = args.L[li + 1].tw[k1];  // in flight while this layer is hashed
        uint32_t m = n, lvl = 0;
        if (k < n) {
            const QMatrix alpha(QM31{{al[0], al[1], al[2], al[3]}});
            const QM31 f = fold_pair({{in[0].x, in[1].x, in[2].x, in[3].x}}, {{in[0].y, in[1].y, in[2].y, in[3].y}},
                                     alpha, tw);
            if (quads) {
                const uint32_t l = tid & 3;
                const uint32_t fl = l == 0 ? f.v[0] : l == 1 ? f.v[1] : l == 2 ? f.v[2] : f.v[3];
                val[l][k] = fl;
                uint32_t* o = l == 0 ? L.out[0] : l == 1 ? L.out[1] : l == 2 ? L.out[2] : L.out[3];
                o[boff + k] = fl;
                uint32_t hl, hh;
                b2s_leaf_quad<4>(f.v, hl, hh);
                qa[8 * k + l] = hl;
                qa[8 * k + 4 + l] = hh;
            } else {
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    val[c][k] = f.v[c];
                    L.out[c][boff + k] = f.v[c];
                }
                uint32_t h[8];
                b2s_leaf4(f.v[0], f.v[1], f.v[2], f.v[3], h);
                if (n > TAIL_QUAD_NODES) {
#pragma unroll
                    for (int q = 0; q < 8; q++) nodes[q * W + k] = h[q];
                } else {
                    store8(qa + 8 * k, h);
                }
            }
        }
        lds_barrier();
        block_lane_levels<W>(nodes, qa, m, lvl, 0, st);
        uint64_t idx0 = 0;
        uint32_t *cur = qa, *nxt = qb;
        block_quad_reduce(cur, nxt, m, lvl, idx0, st);
        // the next layer's inputs, before its values overwrite them
        n /= 2;
        k = k1;
        tw = tw1;
        if (more && k < n) {
#pragma unroll
            for (int c = 0; c < 4; c++) in[c] = *(const uint2*)(&val[c][2 * k]);
        }
        if (tid < 64) {  // one wave: narrow levels and transcript
            uint32_t rl, rh;
            narrow_root(cur, nxt, m, lvl, idx0, st, rl, rh);
            if (tid < 4) {
                L.root_dst[boff + tid] = rl;
                L.root_dst[boff + 4 + tid] = rh;
            }
            tr.mix(rl, rh);
            uint32_t w = 0;
            if (L.alpha_dst && tr.draw(w) && tid < 4) {
                al[tid] = w;
                L.alpha_dst[boff + tid] = w;
            }
        }
        lds_barrier();
    }
    if (tid < 64) tr.store(ch);
}

// Launches fri_tail_kernel over layers [j0, J) (in chunks of FRI_TAIL_MAX_LAYERS);
// layer(j) fills the descriptor of layer j, alpha(j) is the device address of
// its challenge (alpha(j0) already drawn).
template <class LayerFn, class AlphaFn>
void launch_fri_tail(uint32_t j0, uint32_t J, LayerFn&& layer, AlphaFn&& alpha, DevChannel* ch, uint32_t batch,
                     uint64_t bs, hipStream_t s) {
    for (uint32_t j = j0; j < J; j += FRI_TAIL_MAX_LAYERS) {
        FriTailArgs a = {};
        a.n_layers = J - j < FRI_TAIL_MAX_LAYERS ? J - j : FRI_TAIL_MAX_LAYERS;
        for (uint32_t i = 0; i < a.n_layers; i++) {
            a.L[i] = layer(j + i);
            if (a.L[i].n < 2 || a.L[i].n > FRI_TAIL_MAX_ITEMS || (a.L[i].n & (a.L[i].n - 1))) {
                set_error(-2, "fri_tail: layer size out of range");
                return;
            }
        }
        a.alpha0 = alpha(j);
        a.channel = ch;
        fri_tail_kernel<<<dim3(1, batch), FRI_TAIL_THREADS, 0, s>>>(a, bs);
        check_launch("fri_tail_kernel");
    }
}

}  // namespace vx
