// Reference-ABI FRI fold, Fibonacci quotient and zero-pad kernels
// (cuda/fri.cu:10-121, cuda/constraint.cu:10-153). These are the per-call
// entry points the reference prover binds; the fused prover path computes the
// same values inside its commit kernels instead of materialising them.
#include "common.hpp"
#include "field.hpp"

namespace vx {

// All four kernels are bound by device memory (52 bytes a folded value, 20 a
// quotient value). A thread takes one folded value, an 8-byte load of each
// column (two a thread, with 16-byte loads, are slower at most sizes: half of 2^21 line
// 17.7 us, 16.7 so, circle 23.7 and 21.0; 2^24 line 153 and 148; 11 values 0.6 slower by their
// ragged end), or of long arrays four quotient or padded words with 16-byte accesses
// (VEC); a ragged end goes word by word.
struct SoaIn {
    const uint32_t* c[4];
};
struct SoaOut {
    uint32_t* c[4];
};

__global__ __launch_bounds__(256) void fold_line_soa_kernel(SoaIn in, const uint32_t* __restrict__ tw, SoaOut out,
                                                          QM31 alpha, uint32_t half_n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= half_n) return;
    const QMatrix al(alpha);
    QM31 f0, f1;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        f0.v[c] = in.c[c][2ull * i];
        f1.v[c] = in.c[c][2ull * i + 1];
    }
    const QM31 r = fold_pair(f0, f1, al, tw[i]);
#pragma unroll
    for (int c = 0; c < 4; c++) out.c[c][i] = r.v[c];
}

// dst = dst * alpha_sq + fold; the product and the fold's share one reduction.
__device__ __forceinline__ QM31 fold_onto(QM31 prev, QM31 f0, QM31 f1, const QMatrix& al, const QMatrix& sq,
                                          uint32_t tw) {
    uint32_t d[4];
    QM31 r;
#pragma unroll
    for (int k = 0; k < 4; k++) d[k] = mmul(msub(f0.v[k], f1.v[k]), tw);
#pragma unroll
    for (int k = 0; k < 4; k++)
        r.v[k] = madd(madd(f0.v[k], f1.v[k]), reduce64(fold64(al.row(k, d)) + fold64(sq.row(k, prev.v))));
    return r;
}

__global__ __launch_bounds__(256) void fold_circle_soa_kernel(SoaOut dst, SoaIn src, const uint32_t* __restrict__ tw,
                                                            QM31 alpha, QM31 alpha_sq, uint32_t half_n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= half_n) return;
    const QMatrix al(alpha), sq(alpha_sq);
    QM31 f0, f1, prev;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        f0.v[c] = src.c[c][2ull * i];
        f1.v[c] = src.c[c][2ull * i + 1];
        prev.v[c] = dst.c[c][i];
    }
    const QM31 r = fold_onto(prev, f0, f1, al, sq, tw[i]);
#pragma unroll
    for (int c = 0; c < 4; c++) dst.c[c][i] = r.v[c];
}

// Words from which a thread takes four. Below, one a thread has the shorter chain and
// no ragged ends (11 quotients 12.2 us at four, call and wait; 11.65 at one; 2^16 4.05
// and 3.85 back to back; padding to 44 words 11.45 and 11.2); above, wider accesses
// stream faster (2^24 quotients 62 and 78, padding to 2^24 words 12.1 and 20).
constexpr uint32_t QUOTIENT_WIDE_MIN = 1u << 18, PAD_WIDE_MIN = 1u << 19;

// q[i] = alpha * (t[(i+2) mod n] - (t[(i+1) mod n] + t[i]))  (constraint.cu:10-36)
// VEC (n >= 8): four words a thread by 16-byte accesses at any word address.
template <bool VEC>
__global__ __launch_bounds__(256) void quotient_kernel(const uint32_t* __restrict__ t, SoaOut out, QM31 alpha,
                                                     uint32_t offset, uint32_t chunk_n, uint32_t n) {
    const uint32_t li = (blockIdx.x * 256 + threadIdx.x) * (VEC ? 4 : 1);
    if (li >= chunk_n) return;
    if (VEC && chunk_n - li >= 4) {
        const uint32_t i = offset + li;  // i + 3 < n
        const u32x4_any a = *(const u32x4_any*)(t + i);
        const uint32_t e = i + 4 < n ? t[i + 4] : t[0];
        const uint32_t f = n - i > 5 ? t[i + 5] : t[i + 5 - n];
        const uint32_t d[4] = {msub(a.z, madd(a.y, a.x)), msub(a.w, madd(a.z, a.y)), msub(e, madd(a.w, a.z)),
                               msub(f, madd(e, a.w))};
#pragma unroll
        for (int c = 0; c < 4; c++)
            *(u32x4_any*)(out.c[c] + li) = u32x4_any{mmul(alpha.v[c], d[0]), mmul(alpha.v[c], d[1]),
                                                     mmul(alpha.v[c], d[2]), mmul(alpha.v[c], d[3])};
        return;
    }
    for (uint32_t l = li; l < chunk_n && l - li < (VEC ? 4u : 1u); l++) {  // li + 4 may pass 2^32
        const uint32_t i = offset + l;
        // one step at a time, so that every n >= 1 wraps as the reference's remainders do
        const uint32_t i1 = i + 1 == n ? 0u : i + 1, i2 = i1 + 1 == n ? 0u : i1 + 1;
        const uint32_t d = msub(t[i2], madd(t[i1], t[i]));
#pragma unroll
        for (int c = 0; c < 4; c++) out.c[c][l] = mmul(alpha.v[c], d);
    }
}

template <bool VEC>
__global__ __launch_bounds__(256) void zero_pad_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                     uint32_t src_n, uint32_t dst_n) {
    const uint64_t i = (uint64_t)(blockIdx.x * 256ull + threadIdx.x) * (VEC ? 4 : 1);
    if (i >= dst_n) return;
    if (VEC && i + 4 <= dst_n && (i + 4 <= src_n || i >= src_n)) {
        *(uint4*)(dst + i) = i < src_n ? *(const uint4*)(src + i) : make_uint4(0, 0, 0, 0);
        return;
    }
    for (uint64_t k = i; k < dst_n && k < i + (VEC ? 4 : 1); k++) dst[k] = k < src_n ? src[k] : 0u;
}

template <class... T>
static bool aligned(uintptr_t bytes, const T*... p) {
    return (((uintptr_t)p | ...) & (bytes - 1)) == 0;
}

static QM31 q_from_host(const uint32_t* a) { return {{a[0], a[1], a[2], a[3]}}; }

}  // namespace vx

using namespace vx;

extern "C" {

void cuda_fold_line_soa(const uint32_t* in0, const uint32_t* in1, const uint32_t* in2, const uint32_t* in3,
                        const uint32_t* twiddles, uint32_t* out0, uint32_t* out1, uint32_t* out2, uint32_t* out3,
                        const uint32_t* alpha, uint32_t half_n) {
    if (!half_n) return;
    const SoaIn in = {{in0, in1, in2, in3}};
    const SoaOut out = {{out0, out1, out2, out3}};
    fold_line_soa_kernel<<<ceil_div(half_n, 256), 256, 0, current_stream()>>>(in, twiddles, out, q_from_host(alpha), half_n);
    check_launch("cuda_fold_line_soa");
}

void cuda_fold_circle_into_line_soa(uint32_t* dst0, uint32_t* dst1, uint32_t* dst2, uint32_t* dst3,
                                    const uint32_t* src0, const uint32_t* src1, const uint32_t* src2,
                                    const uint32_t* src3, const uint32_t* twiddles, const uint32_t* alpha,
                                    const uint32_t* alpha_sq, uint32_t half_n) {
    if (!half_n) return;
    const SoaIn src = {{src0, src1, src2, src3}};
    const SoaOut dst = {{dst0, dst1, dst2, dst3}};
    fold_circle_soa_kernel<<<ceil_div(half_n, 256), 256, 0, current_stream()>>>(dst, src, twiddles, q_from_host(alpha),
                                                                               q_from_host(alpha_sq), half_n);
    check_launch("cuda_fold_circle_into_line_soa");
}

void cuda_fibonacci_quotient(const uint32_t* trace, uint32_t* out0, uint32_t* out1, uint32_t* out2, uint32_t* out3,
                             const uint32_t* alpha, uint32_t n) {
    cuda_fibonacci_quotient_chunk_stream(trace, out0, out1, out2, out3, alpha, 0, n, n, current_stream());
}
void cuda_fibonacci_quotient_chunk(const uint32_t* trace, uint32_t* out0, uint32_t* out1, uint32_t* out2,
                                   uint32_t* out3, const uint32_t* alpha, uint32_t offset, uint32_t chunk_n,
                                   uint32_t global_n) {
    cuda_fibonacci_quotient_chunk_stream(trace, out0, out1, out2, out3, alpha, offset, chunk_n, global_n,
                                         current_stream());
}
void cuda_fibonacci_quotient_chunk_stream(const uint32_t* trace, uint32_t* out0, uint32_t* out1, uint32_t* out2,
                                          uint32_t* out3, const uint32_t* alpha, uint32_t offset, uint32_t chunk_n,
                                          uint32_t global_n, void* stream) {
    if (!chunk_n) return;
    if (!global_n || (uint64_t)offset + chunk_n > global_n) {
        set_error(-2, "cuda_fibonacci_quotient: need offset + chunk_n <= global_n");
        return;
    }
    const SoaOut out = {{out0, out1, out2, out3}};
    if (chunk_n >= QUOTIENT_WIDE_MIN && global_n >= 8)
        quotient_kernel<true><<<ceil_div(chunk_n, 1024), 256, 0, (hipStream_t)stream>>>(
            trace, out, q_from_host(alpha), offset, chunk_n, global_n);
    else
        quotient_kernel<false><<<ceil_div(chunk_n, 256), 256, 0, (hipStream_t)stream>>>(
            trace, out, q_from_host(alpha), offset, chunk_n, global_n);
    check_launch("cuda_fibonacci_quotient");
}
void cuda_zero_pad(const uint32_t* src, uint32_t* dst, uint32_t src_n, uint32_t dst_n) {
    if (!dst_n) return;
    if (dst_n >= PAD_WIDE_MIN && aligned(16, src, dst))
        zero_pad_kernel<true><<<ceil_div(dst_n, 1024), 256, 0, current_stream()>>>(src, dst, src_n, dst_n);
    else
        zero_pad_kernel<false><<<ceil_div(dst_n, 256), 256, 0, current_stream()>>>(src, dst, src_n, dst_n);
    check_launch("cuda_zero_pad");
}

}  // extern "C"
