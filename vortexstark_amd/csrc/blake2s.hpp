// Blake2s-256 compression for gfx950 (RFC 7693; the reference's single-block
// helper is src/channel.rs:222-298 and its GPU copy cuda/include/blake2s.cuh).
//
// All state lives in VGPRs. Rotations lower to v_alignbit_b32 and the
// three-input adds to v_add3_u32, so one G costs 12 VALU ops; the feed-forward
// is one v_bitop3_b32 per word: a compression is 960 + 8 VALU ops. The round
// schedule is written out with compile-time message indices so no message word
// is ever addressed dynamically.
//
// Issue order. A gfx950 SIMD issues a second VALU instruction of another wave
// beside the one of its first-chosen wave when that second instruction is a
// plain two-operand add, subtract, logic op, right shift or move (measured:
// streams of v_add_u32 / v_xor_b32 / v_bitop3_b32 run at 62-66 T lane-ops/s,
// of v_add3_u32, v_alignbit_b32, v_min_u32 or v_mad_u64_u32 at 30-38 T). The
// first choice goes to the wave of highest priority, then the oldest, so left
// alone the younger waves all come to wait at a rotation or a three-input add
// while the oldest wave owns the SIMD, and nothing pairs: 38 T. The rounds
// below therefore run row-wise over the four G functions (and over K
// independent compressions), with the wave's priority raised for the rows only
// the first slot takes (add3, rotate) and dropped for the rows either slot
// takes (xor, add): a wave at a rotation goes first and another wave's xors
// and adds fill the second slot. Measured on one MI355X, node hashes in a
// loop: 40.1 G/s as single G functions at any occupancy; row-wise with
// priorities 55.8 / 58.0 / 66.1 / 69.9 G/s at 2 / 3 / 4 / 8 waves a SIMD, and
// with two compressions interleaved 59.7 / 60.1 / 68.9 / 69.6 G/s. A lone wave
// a SIMD has nothing to pair with and pays for the s_setprio instructions
// (1.64 -> 2.15 us a compression): PRIO = false, for launches of at most
// LONE_THREADS threads.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "field.hpp"

namespace vx {

constexpr uint32_t B2S_IV0 = 0x6A09E667u, B2S_IV1 = 0xBB67AE85u, B2S_IV2 = 0x3C6EF372u, B2S_IV3 = 0xA54FF53Au;
constexpr uint32_t B2S_IV4 = 0x510E527Fu, B2S_IV5 = 0x9B05688Cu, B2S_IV6 = 0x1F83D9ABu, B2S_IV7 = 0x5BE0CD19u;
// Parameter block word 0: digest length 32, key length 0, fanout 1, depth 1.
constexpr uint32_t B2S_H0 = B2S_IV0 ^ 0x01010020u;

constexpr uint32_t LONE_THREADS = 1u << 16;  // one wave for each SIMD of 256 CUs

#define VX_ROTR(x, n) __builtin_rotateright32((x), (n))
// x ^ y ^ z in one gfx950 instruction (v_bitop3_b32, truth table 0x96)
#define VX_XOR3(x, y, z) __builtin_amdgcn_bitop3_b32((x), (y), (z), 0x96)

// Message schedule of round r (RFC 7693, section 2.7).
constexpr uint8_t B2S_SIGMA[10][16] = {
    {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15}, {14, 10, 4, 8, 9, 15, 13, 6, 1, 12, 0, 2, 11, 7, 5, 3},
    {11, 8, 12, 0, 5, 2, 15, 13, 10, 14, 3, 6, 7, 1, 9, 4}, {7, 9, 3, 1, 13, 12, 11, 14, 2, 6, 5, 10, 4, 0, 15, 8},
    {9, 0, 5, 7, 2, 4, 10, 15, 14, 1, 11, 12, 6, 8, 3, 13}, {2, 12, 6, 10, 0, 11, 8, 3, 4, 13, 7, 5, 15, 14, 1, 9},
    {12, 5, 1, 15, 14, 13, 4, 10, 0, 7, 6, 3, 9, 2, 8, 11}, {13, 11, 7, 14, 12, 1, 3, 9, 5, 0, 15, 4, 8, 6, 2, 10},
    {6, 15, 14, 9, 11, 3, 0, 8, 12, 2, 13, 7, 1, 4, 10, 5}, {10, 2, 8, 4, 7, 6, 1, 5, 15, 11, 9, 14, 3, 12, 13, 0},
};

// Whether a row of additions takes a message word that is not known to be zero
// (words NZ .. 15 are): if not, its adds are two-operand ones.
template <int NZ>
constexpr bool b2s_row_has_word(int r, int j) {
    return B2S_SIGMA[r][j] < NZ || B2S_SIGMA[r][j + 2] < NZ || B2S_SIGMA[r][j + 4] < NZ || B2S_SIGMA[r][j + 6] < NZ;
}

// Half of the G functions of one step of round R, row by row: message words
// sigma[R][J + 2i], rotations R1 and R2; column i of the state takes b, c, d
// rotated by SH, 2 SH, 3 SH columns (SH = 0: columns, 1: diagonals). On entry
// and exit the wave is at priority 1.
template <int K, int NZ, bool PRIO, int R, int J, int SH, int R1, int R2>
__device__ __forceinline__ void b2s_half(uint32_t v[K][16], const uint32_t m[K][16]) {
    constexpr bool WORDS = b2s_row_has_word<NZ>(R, J);
    if (PRIO && !WORDS) VX_PRIO(0);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int k = 0; k < K; k++) v[k][i] = v[k][i] + v[k][4 + ((i + SH) & 3)] + m[k][B2S_SIGMA[R][J + 2 * i]];
    if (PRIO && WORDS) VX_PRIO(0);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int k = 0; k < K; k++) v[k][12 + ((i + 3 * SH) & 3)] ^= v[k][i];
    if (PRIO) VX_PRIO(1);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int k = 0; k < K; k++) v[k][12 + i] = VX_ROTR(v[k][12 + i], R1);
    if (PRIO) VX_PRIO(0);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int k = 0; k < K; k++) v[k][8 + ((i + 2 * SH) & 3)] += v[k][12 + ((i + 3 * SH) & 3)];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int k = 0; k < K; k++) v[k][4 + ((i + SH) & 3)] ^= v[k][8 + ((i + 2 * SH) & 3)];
    if (PRIO) VX_PRIO(1);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int k = 0; k < K; k++) v[k][4 + i] = VX_ROTR(v[k][4 + i], R2);
}
template <int K, int NZ, bool PRIO, int R>
__device__ __forceinline__ void b2s_rounds(uint32_t v[K][16], const uint32_t m[K][16]) {
    if constexpr (R < 10) {
        b2s_half<K, NZ, PRIO, R, 0, 0, 16, 12>(v, m);
        b2s_half<K, NZ, PRIO, R, 1, 0, 8, 7>(v, m);
        b2s_half<K, NZ, PRIO, R, 8, 1, 16, 12>(v, m);
        b2s_half<K, NZ, PRIO, R, 9, 1, 8, 7>(v, m);
        b2s_rounds<K, NZ, PRIO, R + 1>(v, m);
    }
}

// h[k] <- compress(h[k], m[k], t, f) for K independent blocks. Words NZ .. 15
// of every block are zero. m must be indexable with constants only. PRIO =
// false leaves the priorities alone, for waves that have a SIMD to themselves.
template <int K, int NZ, bool PRIO = true>
__device__ __forceinline__ void b2s_compress_n(uint32_t h[K][8], const uint32_t m[K][16], uint32_t t, uint32_t f) {
    uint32_t v[K][16];
#pragma unroll
    for (int k = 0; k < K; k++) {
#pragma unroll
        for (int i = 0; i < 8; i++) v[k][i] = h[k][i];
        v[k][8] = B2S_IV0;
        v[k][9] = B2S_IV1;
        v[k][10] = B2S_IV2;
        v[k][11] = B2S_IV3;
        v[k][12] = B2S_IV4 ^ t;
        v[k][13] = B2S_IV5;
        v[k][14] = B2S_IV6 ^ f;
        v[k][15] = B2S_IV7;
    }
    if (PRIO) VX_PRIO(1);
    b2s_rounds<K, NZ, PRIO, 0>(v, m);
    if (PRIO) VX_PRIO(0);
#pragma unroll
    for (int k = 0; k < K; k++)
#pragma unroll
        for (int i = 0; i < 8; i++) h[k][i] = VX_XOR3(h[k][i], v[k][i], v[k][8 + i]);
}
template <int NZ = 16, bool PRIO = true>
__device__ __forceinline__ void b2s_compress(uint32_t h[8], const uint32_t m[16], uint32_t t, uint32_t f) {
    uint32_t hk[1][8], mk[1][16];
#pragma unroll
    for (int i = 0; i < 8; i++) hk[0][i] = h[i];
#pragma unroll
    for (int i = 0; i < 16; i++) mk[0][i] = m[i];
    b2s_compress_n<1, NZ, PRIO>(hk, mk, t, f);
#pragma unroll
    for (int i = 0; i < 8; i++) h[i] = hk[0][i];
}

__device__ __forceinline__ void b2s_init(uint32_t h[8]) {
    h[0] = B2S_H0;
    h[1] = B2S_IV1;
    h[2] = B2S_IV2;
    h[3] = B2S_IV3;
    h[4] = B2S_IV4;
    h[5] = B2S_IV5;
    h[6] = B2S_IV6;  // no personalisation on any hash of this path (cuda/blake2s.cu:9-10)
    h[7] = B2S_IV7;
}

// Merkle node: H(left || right), t = 64 (cuda/blake2s.cu:65-89).
template <bool PRIO = true>
__device__ __forceinline__ void b2s_node(const uint32_t l[8], const uint32_t r[8], uint32_t out[8]) {
    uint32_t m[16];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        m[i] = l[i];
        m[8 + i] = r[i];
    }
    b2s_init(out);
    b2s_compress<16, PRIO>(out, m, 64u, 0xFFFFFFFFu);
}

// Leaves of N words each (N <= 4, t = 4 N, the Merkle leaf rule of
// cuda/blake2s.cu:45-60 and merkle.rs:538-556), K at once: K = 1, or both leaves of a pair
// with their rounds interleaved (two compressions' rows side by side keep more
// instructions between dependent ones; see the figures above).
template <int K, int N, bool PRIO = true>
__device__ __forceinline__ void b2s_leaves(const uint32_t w[K][N], uint32_t out[K][8]) {
    uint32_t m[K][16];
#pragma unroll
    for (int k = 0; k < K; k++) {
#pragma unroll
        for (int i = 0; i < 16; i++) m[k][i] = i < N ? w[k][i < N ? i : 0] : 0u;
        b2s_init(out[k]);
    }
    b2s_compress_n<K, N, PRIO>(out, m, 4u * N, 0xFFFFFFFFu);
}

// Leaf of one M31 word (single-column trace tree, t = 4).
__device__ __forceinline__ void b2s_leaf1(uint32_t v, uint32_t out[8]) {
    const uint32_t w[1][1] = {{v}};
    uint32_t h[1][8];
    b2s_leaves<1, 1>(w, h);
#pragma unroll
    for (int i = 0; i < 8; i++) out[i] = h[0][i];
}

// Leaf of one QM31 (SoA4 trees, t = 16).
__device__ __forceinline__ void b2s_leaf4(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t out[8]) {
    const uint32_t w[1][4] = {{a, b, c, d}};
    uint32_t h[1][8];
    b2s_leaves<1, 4>(w, h);
#pragma unroll
    for (int i = 0; i < 8; i++) out[i] = h[0][i];
}

// Parent of two leaves of N words.
template <int N, bool PRIO = true>
__device__ __forceinline__ void b2s_leaf_pair(const uint32_t w[2][N], uint32_t out[8]) {
    uint32_t h[2][8];
    if constexpr (PRIO) {
        b2s_leaves<2, N>(w, h);
    } else {  // one after the other: interleaved, a lone wave is slower (2^12 pairs 6.74 us, 6.59 so)
#pragma unroll
        for (int k = 0; k < 2; k++) {
            uint32_t x[1][N], y[1][8];
#pragma unroll
            for (int i = 0; i < N; i++) x[0][i] = w[k][i];
            b2s_leaves<1, N, false>(x, y);
#pragma unroll
            for (int i = 0; i < 8; i++) h[k][i] = y[0][i];
        }
    }
    b2s_node<PRIO>(h[0], h[1], out);
}

// ---------------------------------------------------------------- quad-cooperative form
// Four lanes (a quad: lanes 4q..4q+3 of a wave) compute one compression; lane
// l holds column l of the 4x4 state (v[l], v[4+l], v[8+l], v[12+l]). Used where
// a tree level is too narrow to fill a wave: such a level's time is one lone
// wave's instruction count (about 4 cycles each), which this form cuts from
// about 980 to about 300.
//
// The diagonal step keeps row 1 in place (its rotation ends every half step, so
// it is the one row the next half waits for) and brings rows 0, 2 and 3 over
// from lanes l - 1, l + 1, l + 2; the quad permutes fold into the adds and xors
// that consume the rows (DPP operands), back again in the next column step.
// Lane l then works on diagonal l - 1, so it takes that diagonal's words.

// value from lane (l + k) % 4 of the same quad. A quad permute reads only lanes
// of its own quad, so no lane ever reads an invalid source and bound_ctrl
// changes nothing in the result; set, it lets the compiler fold the move into
// the add or xor that consumes it.
__device__ __forceinline__ uint32_t quad_rot1(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x39, 0xF, 0xF, true);
}
__device__ __forceinline__ uint32_t quad_rot2(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xF, 0xF, true);
}
__device__ __forceinline__ uint32_t quad_rot3(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x93, 0xF, 0xF, true);
}

// mask ? a : b for a mask of all ones or all zeros: one v_bitop3_b32
__device__ __forceinline__ uint32_t b2s_pick(uint32_t mask, uint32_t a, uint32_t b) {
    return __builtin_amdgcn_bitop3_b32(mask, a, b, 0xCA);
}

// Word of sigma[r] that lane l takes as its K-th (0, 1: column step; 2, 3: diagonal step).
__host__ __device__ constexpr int b2s_lane_word(int r, int l, int k) {
    return k < 2 ? B2S_SIGMA[r][2 * l + k] : B2S_SIGMA[r][8 + 2 * ((l + 3) & 3) + (k - 2)];
}

// One round on the lane's words x[0..3]. First half of a step: rows 0, 2, 3
// come from the lanes of the previous step's alignment.
template <bool FIRST>
__device__ __forceinline__ void b2s_quad_round(const uint32_t x[4], uint32_t& a, uint32_t& b, uint32_t& c,
                                               uint32_t& d) {
    if (FIRST) {
        a = a + b + x[0];
        d ^= a;
    } else {
        a = quad_rot1(a) + x[0] + b;
        d = quad_rot2(d) ^ a;
    }
    d = VX_ROTR(d, 16);
    c = (FIRST ? c : quad_rot3(c)) + d;
    b = VX_ROTR(b ^ c, 12);
    a = a + b + x[1];
    d = VX_ROTR(d ^ a, 8);
    c += d;
    b = VX_ROTR(b ^ c, 7);
    a = quad_rot3(a) + x[2] + b;
    d = VX_ROTR(quad_rot2(d) ^ a, 16);
    c = quad_rot1(c) + d;
    b = VX_ROTR(b ^ c, 12);
    a = a + b + x[3];
    d = VX_ROTR(d ^ a, 8);
    c += d;
    b = VX_ROTR(b ^ c, 7);
}
__device__ __forceinline__ void b2s_quad_start(uint32_t t, uint32_t f, uint32_t& c, uint32_t& d) {
    const uint32_t l = threadIdx.x & 3;
    const uint32_t m0 = 0u - (l & 1u), m1 = 0u - ((l >> 1) & 1u);
    c = b2s_pick(m1, b2s_pick(m0, B2S_IV3, B2S_IV2), b2s_pick(m0, B2S_IV1, B2S_IV0));
    d = b2s_pick(m1, b2s_pick(m0, B2S_IV7, B2S_IV6 ^ f), b2s_pick(m0, B2S_IV5, B2S_IV4 ^ t));
}
// Feed-forward; rows 0, 2, 3 leave the last diagonal step's alignment.
__device__ __forceinline__ void b2s_quad_finish(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t& hl,
                                                uint32_t& hh) {
    hl = VX_XOR3(hl, quad_rot1(a), quad_rot3(c));
    hh = VX_XOR3(hh, b, quad_rot2(d));
}

// Message word b2s_lane_word(R, l, K) of quad lane l, chosen among the four
// candidates with the lane's bit masks (m0: bit 0 of l set, m1: bit 1).
template <int R, int K>
__device__ __forceinline__ uint32_t b2s_quad_word(const uint32_t m[16], uint32_t m0, uint32_t m1) {
    constexpr int w0 = b2s_lane_word(R, 0, K), w1 = b2s_lane_word(R, 1, K), w2 = b2s_lane_word(R, 2, K),
                  w3 = b2s_lane_word(R, 3, K);
    return b2s_pick(m1, b2s_pick(m0, m[w3], m[w2]), b2s_pick(m0, m[w1], m[w0]));
}
template <int R>
__device__ __forceinline__ void b2s_quad_rounds(const uint32_t m[16], uint32_t m0, uint32_t m1, uint32_t& a,
                                                uint32_t& b, uint32_t& c, uint32_t& d) {
    if constexpr (R < 10) {
        const uint32_t x[4] = {b2s_quad_word<R, 0>(m, m0, m1), b2s_quad_word<R, 1>(m, m0, m1),
                               b2s_quad_word<R, 2>(m, m0, m1), b2s_quad_word<R, 3>(m, m0, m1)};
        b2s_quad_round<R == 0>(x, a, b, c, d);
        b2s_quad_rounds<R + 1>(m, m0, m1, a, b, c, d);
    }
}

// Lane l: in hl = h[l], hh = h[4+l]; out the same words of the new chaining value.
// Every lane of the quad holds all 16 message words and picks those of its G
// functions by selects, which issue in the shadow of the rounds' dependent chain.
// All four lanes of the quad must be active.
__device__ __forceinline__ void b2s_compress_quad_words(const uint32_t m[16], uint32_t t, uint32_t f, uint32_t& hl,
                                                        uint32_t& hh) {
    const uint32_t l = threadIdx.x & 3;
    const uint32_t m0 = 0u - (l & 1u), m1 = 0u - ((l >> 1) & 1u);
    uint32_t a = hl, b = hh, c, d;
    b2s_quad_start(t, f, c, d);
    b2s_quad_rounds<0>(m, m0, m1, a, b, c, d);
    b2s_quad_finish(a, b, c, d, hl, hh);
}
// The same with the quad's message in memory, read before the first round, so no
// LDS access waits inside the chain.
__device__ __forceinline__ void b2s_compress_quad(const uint32_t* msg, uint32_t t, uint32_t f, uint32_t& hl,
                                                  uint32_t& hh) {
    uint32_t m[16];
#pragma unroll
    for (int i = 0; i < 16; i++) m[i] = msg[i];  // two words a read: 16-byte reads deliver later
    b2s_compress_quad_words(m, t, f, hl, hh);
}
// Message words 4 j .. 4 j + 3 of a quad from word 4 j + l in lane l.
__device__ __forceinline__ void quad_gather(uint32_t x, uint32_t m[4]) {
    m[0] = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x00, 0xF, 0xF, true);
    m[1] = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x55, 0xF, 0xF, true);
    m[2] = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xAA, 0xF, 0xF, true);
    m[3] = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xFF, 0xF, 0xF, true);
}
// Initial chaining words of lane l (IV with the parameter block folded in).
__device__ __forceinline__ void b2s_quad_init(uint32_t& hl, uint32_t& hh) {
    const uint32_t l = threadIdx.x & 3;
    hl = l == 0 ? B2S_H0 : l == 1 ? B2S_IV1 : l == 2 ? B2S_IV2 : B2S_IV3;
    hh = l == 0 ? B2S_IV4 : l == 1 ? B2S_IV5 : l == 2 ? B2S_IV6 : B2S_IV7;
}

// Leaf of N words (N <= 4, t = 4 N), quad-cooperatively; every lane of the quad
// holds all of w. Words N .. 15 are zero, so of a round's sixteen words few
// are not: each word is kept masked per lane, and a lane's word of a round is
// the or of the (mostly one or no) masked words that can land there.
template <int N, int R, int K>
__device__ __forceinline__ uint32_t b2s_leaf_word(const uint32_t mk[N][4]) {
    uint32_t x = 0;
#pragma unroll
    for (int l = 0; l < 4; l++) {
        const int w = b2s_lane_word(R, l, K);
        if (w < N) x |= mk[w < N ? w : 0][l];
    }
    return x;
}
template <int N, int R>
__device__ __forceinline__ void b2s_leaf_quad_rounds(const uint32_t mk[N][4], uint32_t& a, uint32_t& b, uint32_t& c,
                                                     uint32_t& d) {
    if constexpr (R < 10) {
        const uint32_t x[4] = {b2s_leaf_word<N, R, 0>(mk), b2s_leaf_word<N, R, 1>(mk), b2s_leaf_word<N, R, 2>(mk),
                               b2s_leaf_word<N, R, 3>(mk)};
        b2s_quad_round<R == 0>(x, a, b, c, d);
        b2s_leaf_quad_rounds<N, R + 1>(mk, a, b, c, d);
    }
}
template <int N>
__device__ __forceinline__ void b2s_leaf_quad(const uint32_t w[N], uint32_t& hl, uint32_t& hh) {
    const uint32_t l = threadIdx.x & 3;
    uint32_t mk[N][4];
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) mk[i][k] = l == k ? w[i] : 0u;
    b2s_quad_init(hl, hh);
    uint32_t a = hl, b = hh, c, d;
    b2s_quad_start(4u * N, 0xFFFFFFFFu, c, d);
    b2s_leaf_quad_rounds<N, 0>(mk, a, b, c, d);
    b2s_quad_finish(a, b, c, d, hl, hh);
}

}  // namespace vx
