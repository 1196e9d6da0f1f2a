// bf16 / fp32 activations into the fp16 rows every matmul and gather kernel
// reads, without losing range:
//
//   x16[r][k] = fp16(x[r][k] * 2^-e[r]),   e[r] = E - 15 where max_k |x[r][k]| = f 2^E, f in [0.5, 1)
//
// so each row's largest magnitude lands in [2^14, 2^15) (below fp16's 65504)
// and the kernels multiply their fp32 results by 2^e[r] before any bias or
// activation (ldexp: exact).  A bf16 value keeps all its bits (8-bit mantissa
// inside fp16's 11) unless it lies more than 2^29 below its row's maximum,
// where fp16 turns subnormal; such entries add at most 2^-29 of the largest
// term each.  An fp32 value rounds once to 11 bits, as before, but no longer
// overflows past 65504 or flushes below 2^-14.  Rows of zeros get e = 0; inf
// and NaN pass through (e = 0 for a row whose maximum is not finite).
//
// This replaces the reference's convert-on-load of bf16 / fp32 operands
// (accumulate in fp32, gmlx/dtypes.py:8-9, 16-17, 26-29): the MFMA path of
// these kernels takes fp16 operands, and the per-row power of two keeps the
// conversion exact for bf16.
#include "kq_common.h"

namespace {

// 8 consecutive activations as fp32: one 16-byte load (bf16) or two (fp32).
template <int XT>
struct Chunk {
    u32x4 w[XT == 2 ? 2 : 1];

    __device__ __forceinline__ void load(const char *row, int c) {
#pragma unroll
        for (int i = 0; i < (XT == 2 ? 2 : 1); ++i) w[i] = *(const u32x4 *)(row + (int64_t)c * (XT == 2 ? 32 : 16) + 16 * i);
    }
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int i = 0; i < (XT == 2 ? 2 : 1); ++i) w[i] = u32x4{0u, 0u, 0u, 0u};
    }
    __device__ __forceinline__ float value(int i) const {
        // (a value of its own: bit_cast of a vector element reads element 0)
        const uint32_t u = w[XT == 2 ? i >> 2 : 0][XT == 2 ? i & 3 : i >> 1];
        return __builtin_bit_cast(float, XT == 2 ? u : (i & 1) ? u & 0xFFFF0000u : u << 16);
    }
    __device__ __forceinline__ float largest(float mx) const {
#pragma unroll
        for (int i = 0; i < 8; ++i) mx = fmaxf(mx, fabsf(value(i)));
        return mx;
    }
    __device__ __forceinline__ half8_t scaled(int e) const {
        half8_t h;
#pragma unroll
        for (int i = 0; i < 8; ++i) h[i] = (_Float16)ldexpf(value(i), -e);
        return h;
    }
};

// LANES lanes take a row (a whole workgroup of 512 threads, or one wave of
// it): the row's maximum magnitude, then the scaled fp16 row.  A lane keeps up
// to kHeld chunks of 8 values in registers between the two (rows of up to
// 16384 per workgroup, 2048 per wave), so the row is read once, 16 bytes a
// lane; longer rows read the rest again.  Bound by latency at decode widths (a
// load, the reduction, a store) and by HBM at prompt widths.  Rows of up to
// 2048 values go one to a wave, eight to a workgroup: they leave most lanes of
// a whole workgroup idle.  Against one workgroup of 256 threads a row loading
// one value each a step and keeping none (us a launch, bf16, rocprofv3): 37
// rows of 4096 (three of four) and 12288, 13.9 -> 4.8; 2048 rows of the same,
// 23.1 -> 12.7; 500 rows of 2048 and 4000 of 768, 7.4 -> 5.2.
constexpr int kThreads = 512, kHeld = 4;

template <int XT, int LANES>
__global__ __launch_bounds__(kThreads) void prepare_rows_kernel(const char *x, int64_t stride_bytes, int rows, int K,
                                                                kq_half *x16, int32_t *e_out) {
    __shared__ float part[kThreads / 64];
    const int lane = (int)threadIdx.x % LANES;
    const int r = (int)blockIdx.x * (kThreads / LANES) + (int)threadIdx.x / LANES;
    if (LANES == 64 && r >= rows) return;  // uniform over the wave; this form has no barrier
    const char *row = x + (int64_t)r * stride_bytes;
    const int n = K / 8;
    Chunk<XT> held[kHeld];
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < kHeld; ++i) {
        const int c = lane + LANES * i;
        if (c < n) held[i].load(row, c);
        else held[i].zero();
    }
#pragma unroll
    for (int i = 0; i < kHeld; ++i) mx = held[i].largest(mx);
    for (int c = lane + LANES * kHeld; c < n; c += LANES) {
        Chunk<XT> v;
        v.load(row, c);
        mx = v.largest(mx);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if constexpr (LANES > 64) {
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = mx;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kThreads / 64; ++i) mx = fmaxf(mx, part[i]);
    }
    int e = 0;
    if (mx > 0.f && mx <= 3.402823466e38f) {
        int E;
        (void)frexpf(mx, &E);
        e = E - 15;
    }
    if (lane == 0) e_out[r] = e;
    half8_t *dst = (half8_t *)(x16 + (int64_t)r * K);
#pragma unroll
    for (int i = 0; i < kHeld; ++i) {
        const int c = lane + LANES * i;
        if (c < n) dst[c] = held[i].scaled(e);
    }
    for (int c = lane + LANES * kHeld; c < n; c += LANES) {
        Chunk<XT> v;
        v.load(row, c);
        dst[c] = v.scaled(e);
    }
}

template <int XT>
void launch_prepare(const void *x, int64_t stride_bytes, int rows, int K, kq_half *x16, int32_t *e, hipStream_t s) {
    constexpr int per = kThreads / 64;
    if (K <= 64 * kHeld * 8)
        hipLaunchKernelGGL((prepare_rows_kernel<XT, 64>), dim3((rows + per - 1) / per), dim3(kThreads), 0, s,
                           (const char *)x, stride_bytes, rows, K, x16, e);
    else
        hipLaunchKernelGGL((prepare_rows_kernel<XT, kThreads>), dim3(rows), dim3(kThreads), 0, s, (const char *)x,
                           stride_bytes, rows, K, x16, e);
}

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

}  // namespace

size_t kq_prepared_bytes(int64_t rows, int64_t K) {
    return align256((size_t)rows * (size_t)K * 2) + align256((size_t)rows * 4);
}

// rows x K activations of x_dtype (bf16 or fp32), x_stride elements apart ->
// fp16 rows (K apart) at `out` and their exponents right after
// (kq_prepared_bytes(rows, K) bytes, 256-aligned parts).
int kq_prepare_rows(const void *x, int x_dtype, int64_t x_stride, int32_t rows, int32_t K, void *out,
                    const int32_t **exp_out, const void **x16_out, hipStream_t s) {
    kq_half *x16 = (kq_half *)out;
    int32_t *e = (int32_t *)((char *)out + align256((size_t)rows * (size_t)K * 2));
    *x16_out = x16;
    *exp_out = e;
    if (rows <= 0) return KQ_OK;
    if (x_dtype == KQ_DTYPE_F32) launch_prepare<2>(x, x_stride * 4, rows, K, x16, e, s);
    else launch_prepare<1>(x, x_stride * 2, rows, K, x16, e, s);
    return hipGetLastError() == hipSuccess ? KQ_OK : KQ_ERR_LAUNCH_FAILED;
}
