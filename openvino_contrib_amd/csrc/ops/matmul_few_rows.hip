// Products of few activation rows -- up to six, up to 16 on small weights -- with a weight matrix stored [n, k], the
// projections of a decode step of few sequences, on v_mfma_f32_16x16x32 with fp32 accumulation, instead of the library's kernels.
//
// What bounds it: the weights, read once.  A workgroup takes 16 weight rows and its eight wavefronts an eighth of k each;
// a lane's loads are the matrix operands as they stand (weight row lane % 16, eight k of quarter lane / 16; activations
// alike, only the rows that exist), four steps multiplied while the next four are on their way.  No operand passes through
// LDS, where only the eight partial sums meet.  (Loads marked as not to be kept fetch each 128-byte line twice: 52 against
// 43 us at n 28,672; two tiles of weight rows to a workgroup: 53.)
// Measured (bf16, 4 rows, weights from HBM; library -> this): n 28,672 k 4,096: 49.0 -> 44.2 us (5.3 TB/s); 4,096 x 14,336:
// 25.5 -> 22.7; 4,096 x 4,096: 10.3 -> 8.5; 1,024 x 4,096: 10.1 -> 7.1; 512 x 2,048: 9.9 -> 4.7.
#include "ops/ops_common.hpp"

namespace hipops {

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

constexpr int kWaves = 8, kGroup = 4;

template <bool kBf16>
__device__ __forceinline__ float4_t mma(uint4_t a, uint4_t b, float4_t c) {
    if constexpr (kBf16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
}
template <bool kBf16>
__device__ __forceinline__ uint32_t cvt2(float lo, float hi) {
    if constexpr (kBf16)
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2_t){lo, hi}, bf16x2_t));
    else
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2_t){lo, hi}, half2_t));
}

// a [m, k], b [n, k], c [m, n] (of the operands' type, or fp32); steps = k / 32.
template <bool kBf16>
__global__ __launch_bounds__(64 * kWaves) void matmul_few_rows_kernel(const uint16_t* a, const uint16_t* b, void* c, int m, int n, int64_t k, int steps,
                                                                      int c_is_f32) {
    __shared__ float4_t sums[kWaves][64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, row = lane & 15, quarter = lane >> 4;
    const int n0 = 16 * (int)blockIdx.x;
    const int first = (int)((int64_t)steps * wave / kWaves), last = (int)((int64_t)steps * (wave + 1) / kWaves);
    const uint16_t* const w = b + (int64_t)min(n0 + row, n - 1) * k + 8 * quarter;
    const uint16_t* const x = a + (int64_t)min(row, m - 1) * k + 8 * quarter;
    const bool real = row < m;
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    struct Group {
        uint4_t w[kGroup], x[kGroup];
    } now, next;
    const auto load = [&](Group& g, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kGroup; u++) g.w[u] = *(const uint4_t*)(w + 32 * (int64_t)min(s + u, last - 1));  // (past the end: unused)
        if (real) {
#pragma unroll
            for (int u = 0; u < kGroup; u++) g.x[u] = *(const uint4_t*)(x + 32 * (int64_t)min(s + u, last - 1));
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const auto multiply = [&](const Group& g, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kGroup; u++)
            if (s + u < last) acc = mma<kBf16>(g.w[u], g.x[u], acc);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int u = 0; u < kGroup; u++) now.x[u] = next.x[u] = (uint4_t){0u, 0u, 0u, 0u};  // (lanes without a row keep these)
    if (first < last) {
        load(now, first);
        for (int s = first; s < last; s += 2 * kGroup) {
            if (s + kGroup < last) load(next, s + kGroup);
            multiply(now, s);
            if (s + 2 * kGroup < last) load(now, s + 2 * kGroup);
            multiply(next, s + kGroup);
        }
    }
    // register r: weight row 4 quarter + r of the tile, activation row lane % 16
    sums[wave][lane] = acc;
    __syncthreads();
    if (wave != 0) return;
    float4_t sum = sums[0][lane];
#pragma unroll
    for (int i = 1; i < kWaves; i++) sum += sums[i][lane];
    const int at = n0 + 4 * quarter;  // (n is a multiple of 4)
    if (!real || at >= n) return;
    if (c_is_f32)
        *(float4_t*)((float*)c + (int64_t)row * n + at) = sum;
    else
        *(uint2_t*)((uint16_t*)c + (int64_t)row * n + at) = (uint2_t){cvt2<kBf16>(sum[0], sum[1]), cvt2<kBf16>(sum[2], sum[3])};
}

}  // namespace

// 16-bit operands, one matrix, the weights' rows along k, whole steps of k, 16-byte aligned rows.
// Every activation row costs load instructions of its own and the library's kernels, built for tiles of 16, do not mind them,
// so it is up to 6 rows, or 16 where the weights are small enough for the launch to be most of the time (library -> this,
// 16 rows: 512 x 2,048 10.1 -> 5.6 us, 1,024 x 4,096 10.0 -> 9.1, 4,096 x 4,096 10.2 -> 10.6; 8 rows: 3,072 x 8,192 14.0 -> 14.6), and
// up to 4 on the largest (128,256 x 4,096, 1 / 4 / 6 rows: 173 / 174 / 175 -> 166 / 175 / 184).
// A wavefront goes through its eighth of k alone, so k must not be long where n is short: a chain of 6,144 takes as long as the
// library's split one (4 rows: 512 x 6,144 10.2 -> 9.6, 16 x 6,144 9.9 -> 9.1, but 64 x 8,192 10.1 -> 11.8, 256 x 16,384 13.3 -> 21.9;
// 16 rows: 512 x 6,144 11.0 -> 12.5), beyond it n bounds k (2,048 x 7,168 12.4 -> 11.1, 4,096 x 14,336 25.5 -> 22.3,
// but 2,048 x 8,192 12.0 -> 12.7, 3,072 x 12,288 19.0 -> 19.4, 4,096 x 16,384 29.8 -> 34.4, 8,192 x 28,672 85.1 -> 87.0).
// Large weights only where every wavefront's k is whole rounds of two groups (4 rows: 8,192 x 4,096 15.8 -> 15.2, 14,336 x
// 2,048 15.6 -> 15.1, but 21,504 x 3,072 27.4 -> 28.9 and 5,120 x 5,120 16.1 -> 17.1).
bool matmul_few_rows_supported(const hipops_matmul_desc* d, const void* a, const void* b, const void* c) {
    const auto aligned16 = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
    const int64_t weights = d->n * d->k;
    if ((d->ab_dtype != HIPATTN_F16 && d->ab_dtype != HIPATTN_BF16) || d->batch != 1 || d->transpose_a || !d->transpose_b || d->n % 4 != 0 ||
        d->k % 32 != 0 || !aligned16(a) || !aligned16(b) || !aligned16(c))
        return false;
    if (d->m > 6) return d->m <= 16 && weights <= (1 << 22) && d->k <= 4096;
    if (d->m > 4 && weights > (1 << 27)) return false;
    if (d->k > 6144 && (2 * d->k > 7 * d->n || weights > (1 << 27))) return false;
    return weights <= (1 << 24) || d->k % (2 * 32 * kGroup * kWaves) == 0;
}

hipattn_status matmul_few_rows(const hipops_matmul_desc* d, const void* a, const void* b, void* c, hipStream_t stream) {
    const dim3 grid((unsigned)((d->n + 15) / 16)), block(64 * kWaves);
    const auto kernel = d->ab_dtype == HIPATTN_BF16 ? matmul_few_rows_kernel<true> : matmul_few_rows_kernel<false>;
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, (const uint16_t*)a, (const uint16_t*)b, c, (int)d->m, (int)d->n, d->k, (int)(d->k / 32),
                       d->c_dtype == HIPATTN_F32 ? 1 : 0);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return fail(HIPATTN_HIP_ERROR, "matmul: %s", hipGetErrorString(e));
    return HIPATTN_OK;
}

}  // namespace hipops
