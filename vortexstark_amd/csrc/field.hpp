// M31 / CM31 / QM31 arithmetic for gfx950 device code.
//
// Semantics follow the reference field tower exactly (canonical u32 in [0, p),
// p = 2^31 - 1): src/field/m31.rs:24-121, cm31.rs:78-87, qm31.rs:114-132 and
// cuda/include/{m31,cm31,qm31}.cuh. The instruction choices are CDNA-specific:
// the canonical reduction of r in [0, 2p) is min(r, r - p) (v_sub + v_min_u32,
// no compare/select), and the 62-bit product is folded with one v_alignbit.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vx {

constexpr uint32_t P = 0x7FFFFFFFu;

// Pointers into device memory. A pointer that a kernel reads from memory (a
// column table's) is otherwise generic, and a generic access also occupies the
// LDS path and is waited for with the LDS accesses.
typedef __attribute__((address_space(1))) uint32_t gu32;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) u32x2 gu32x2;
typedef __attribute__((address_space(1))) u32x4 gu32x4;
__device__ __forceinline__ const gu32* as_global(const uint32_t* p) { return (const gu32*)p; }
__device__ __forceinline__ gu32* as_global(uint32_t* p) { return (gu32*)p; }

// Workgroup barrier that orders LDS accesses only. __syncthreads also waits
// for the block's outstanding device-memory stores, which a chain of levels
// that never reads them back would wait for once a level.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Wave priority p from here on, with the instructions before and after kept on
// their side of it. A SIMD issues a second wave's two-operand adds, subtracts,
// logic ops, right shifts and moves beside the instruction of its first-chosen
// wave (highest priority, then oldest), so a wave raises its priority for the
// instructions only the first slot takes (v_add3, v_alignbit, v_min, v_mad_u64,
// other multiplies) and drops it for the rest; left alone, the younger waves
// all come to wait at one of the former and nothing pairs.
#define VX_PRIO(p)                            \
    do {                                      \
        __builtin_amdgcn_sched_barrier(0);    \
        __builtin_amdgcn_s_setprio(p);        \
        __builtin_amdgcn_sched_barrier(0);    \
    } while (0)

// r in [0, 2p) -> r mod p.
__device__ __forceinline__ uint32_t canon(uint32_t r) { return min(r, r - P); }

__device__ __forceinline__ uint32_t madd(uint32_t a, uint32_t b) { return canon(a + b); }
__device__ __forceinline__ uint32_t msub(uint32_t a, uint32_t b) { return canon(a + (P - b)); }
__device__ __forceinline__ uint32_t mneg(uint32_t a) { return a == 0 ? 0 : P - a; }
__device__ __forceinline__ uint32_t mdbl(uint32_t a) { return canon(a << 1); }

__device__ __forceinline__ uint32_t mmul(uint32_t a, uint32_t b) {
    uint64_t p = (uint64_t)a * b;
    uint32_t lo = (uint32_t)p, hi = (uint32_t)(p >> 32);
    // p mod (2^31 - 1) = (p & p31) + (p >> 31); the sum is < 2p for canonical inputs.
    uint32_t top = __builtin_amdgcn_alignbit(hi, lo, 31);
    return canon((lo & P) + top);
}

__device__ __forceinline__ uint32_t mpow(uint32_t b, uint32_t e) {
    uint32_t r = 1;
    while (e) {
        if (e & 1) r = mmul(r, b);
        b = mmul(b, b);
        e >>= 1;
    }
    return r;
}
__device__ __forceinline__ uint32_t msqr_n(uint32_t a, int n) {
    for (int i = 0; i < n; i++) a = mmul(a, a);
    return a;
}
// a^(p-2) = a^(2^31 - 3) by an addition chain: x_k = a^(2^k - 1) from
// x_1, x_2, x_4, x_8, x_16, x_24, x_28, x_29, then x_29^4 * a
// (30 squarings and 8 products, against 61 for square-and-multiply). 0 -> 0.
__device__ __forceinline__ uint32_t minv(uint32_t a) {
    const uint32_t x2 = mmul(mmul(a, a), a);
    const uint32_t x4 = mmul(msqr_n(x2, 2), x2);
    const uint32_t x8 = mmul(msqr_n(x4, 4), x4);
    const uint32_t x16 = mmul(msqr_n(x8, 8), x8);
    const uint32_t x24 = mmul(msqr_n(x16, 8), x8);
    const uint32_t x28 = mmul(msqr_n(x24, 4), x4);
    const uint32_t x29 = mmul(mmul(x28, x28), a);
    return mmul(msqr_n(x29, 2), a);
}

struct CM31 {
    uint32_t a, b;
};
__device__ __forceinline__ CM31 cadd(CM31 x, CM31 y) { return {madd(x.a, y.a), madd(x.b, y.b)}; }
__device__ __forceinline__ CM31 csub(CM31 x, CM31 y) { return {msub(x.a, y.a), msub(x.b, y.b)}; }
// (a + bi)(c + di) with three products: the imaginary part is
// (a + b)(c + d) - ac - bd (Karatsuba; equal to ad + bc mod p).
__device__ __forceinline__ CM31 cmul(CM31 x, CM31 y) {
    const uint32_t ac = mmul(x.a, y.a), bd = mmul(x.b, y.b);
    const uint32_t s = mmul(madd(x.a, x.b), madd(y.a, y.b));
    return {msub(ac, bd), msub(msub(s, ac), bd)};
}

// x < 2^64 -> a value < 2^34 congruent to it mod p (2^32 = 2): one
// v_mad_u64_u32. Four products of canonical values still fit on top of it:
// 4 (p - 1)^2 + 2^34 = 2^64 - 2^35 + 16 + 2^34.
__device__ __forceinline__ uint64_t fold64(uint64_t x) { return (uint64_t)(uint32_t)(x >> 32) * 2u + (uint32_t)x; }
// x < 2^64 -> x mod p
__device__ __forceinline__ uint32_t reduce64(uint64_t x) {
    const uint64_t y = fold64(x);
    return canon(((uint32_t)y & P) + __builtin_amdgcn_alignbit((uint32_t)(y >> 32), (uint32_t)y, 31));
}

// QM31 = a + b*u with u^2 = 2 + i; stored as {a.a, a.b, b.a, b.b}.
struct QM31 {
    uint32_t v[4];
};
__device__ __forceinline__ QM31 qadd(QM31 x, QM31 y) {
    return {{madd(x.v[0], y.v[0]), madd(x.v[1], y.v[1]), madd(x.v[2], y.v[2]), madd(x.v[3], y.v[3])}};
}
__device__ __forceinline__ QM31 qsub(QM31 x, QM31 y) {
    return {{msub(x.v[0], y.v[0]), msub(x.v[1], y.v[1]), msub(x.v[2], y.v[2]), msub(x.v[3], y.v[3])}};
}
__device__ __forceinline__ QM31 qmul_m31(QM31 x, uint32_t s) {
    return {{mmul(x.v[0], s), mmul(x.v[1], s), mmul(x.v[2], s), mmul(x.v[3], s)}};
}
// (A + Bu)(C + Du) = (AC + (2 + i) BD) + ((A + B)(C + D) - AC - BD) u: three
// CM31 products (nine M31 products) instead of four (sixteen).
__device__ __forceinline__ QM31 qmul(QM31 x, QM31 y) {
    const CM31 xa = {x.v[0], x.v[1]}, xb = {x.v[2], x.v[3]};
    const CM31 ya = {y.v[0], y.v[1]}, yb = {y.v[2], y.v[3]};
    const CM31 ac = cmul(xa, ya), bd = cmul(xb, yb);
    const CM31 s = cmul(cadd(xa, xb), cadd(ya, yb));
    // bd * (2 + i) = (2p - q) + (p + 2q) i
    const CM31 bdu = {msub(mdbl(bd.a), bd.b), madd(bd.a, mdbl(bd.b))};
    const CM31 ra = cadd(ac, bdu), rb = csub(csub(s, ac), bd);
    return {{ra.a, ra.b, rb.a, rb.b}};
}

// Multiplication by a QM31 constant as a 4 x 4 matrix over M31: row k of the
// product alpha * d is sum_j m[k][j] d_j, four products and one reduction, where
// the three-product form takes nine products and some forty additions.
struct QMatrix {
    uint32_t m[4][4];
    __device__ __forceinline__ explicit QMatrix(QM31 a) {
        const uint32_t a0 = a.v[0], a1 = a.v[1], a2 = a.v[2], a3 = a.v[3];
        const uint32_t t = msub(mdbl(a2), a3), s = madd(mdbl(a3), a2);  // 2 a2 - a3, 2 a3 + a2
        m[0][0] = a0, m[0][1] = mneg(a1), m[0][2] = t, m[0][3] = mneg(s);
        m[1][0] = a1, m[1][1] = a0, m[1][2] = s, m[1][3] = t;
        m[2][0] = a2, m[2][1] = mneg(a3), m[2][2] = a0, m[2][3] = mneg(a1);
        m[3][0] = a3, m[3][1] = a2, m[3][2] = a1, m[3][3] = a0;
    }
    __device__ __forceinline__ uint64_t row(int k, const uint32_t d[4]) const {  // < 2^64
        uint64_t x = (uint64_t)m[k][0] * d[0];
        x += (uint64_t)m[k][1] * d[1];
        x += (uint64_t)m[k][2] * d[2];
        x += (uint64_t)m[k][3] * d[3];
        return x;
    }
};

// FRI fold of one pair: (f0 + f1) + alpha * ((f0 - f1) * tw)   (cuda/fri.cu:26-33)
__device__ __forceinline__ QM31 fold_pair(QM31 f0, QM31 f1, const QMatrix& alpha, uint32_t tw) {
    uint32_t d[4];
    QM31 r;
#pragma unroll
    for (int k = 0; k < 4; k++) d[k] = mmul(msub(f0.v[k], f1.v[k]), tw);
#pragma unroll
    for (int k = 0; k < 4; k++) r.v[k] = madd(madd(f0.v[k], f1.v[k]), reduce64(alpha.row(k, d)));
    return r;
}

// Circle group (src/circle.rs:33-39)
struct CPt {
    uint32_t x, y;
};
__device__ __forceinline__ CPt cpmul(CPt p, CPt q) {
    return {msub(mmul(p.x, q.x), mmul(p.y, q.y)), madd(mmul(p.x, q.y), mmul(p.y, q.x))};
}
// initial * step^e by square-and-multiply.
__device__ __forceinline__ CPt cp_pow_mul(CPt initial, CPt step, uint32_t e) {
    CPt r = {1, 0};
    while (e) {
        if (e & 1) r = cpmul(r, step);
        step = cpmul(step, step);
        e >>= 1;
    }
    return cpmul(initial, r);
}

__device__ __forceinline__ uint32_t brev_bits(uint32_t x, uint32_t bits) {
    return bits == 0 ? 0u : (__builtin_bitreverse32(x) >> (32 - bits));
}

// Words every lane reads alike, constant while the kernel runs: scalar loads.
typedef const __attribute__((address_space(4))) uint32_t ConstU32;
typedef const __attribute__((address_space(4))) uint64_t ConstU64;
typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(4)));  // any word address
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(4)));
// words i .. i + RUN - 1 of an array of len words
template <uint32_t RUN>
__device__ __forceinline__ void store_run(uint32_t* out, uint64_t i, uint64_t len, const uint32_t (&w)[RUN]) {
    if (i + RUN <= len) {
#pragma unroll
        for (uint32_t r = 0; r < RUN; r += 4) {
            const u32x4_any v = {w[r], w[r + 1], w[r + 2], w[r + 3]};
            *(__attribute__((address_space(1))) u32x4_any*)(out + i + r) = v;
        }
    } else {
#pragma unroll
        for (uint32_t r = 0; r < RUN; r++)
            if (i + r < len) out[i + r] = w[r];
    }
}

}  // namespace vx
