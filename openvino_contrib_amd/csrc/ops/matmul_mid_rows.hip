// Products of 7 to 64 activation rows with a weight matrix stored [n, k] -- the projections of a decode step of a serving batch -- on
// v_mfma_f32_16x16x32 with fp32 accumulation, instead of the library's kernels.
//
// What bounds it: the weights, read once from HBM.  A workgroup takes 16 weight rows to a wavefront, four or six wavefronts, and a part
// of k; weights and activations come to LDS 64 elements of k at a time (global_load_lds, a ring of kRing stages, one barrier to a stage),
// because the matrix operands as they stand are not what a compute unit loads well: sixteen lanes in sixteen rows take
// 64 clocks to an instruction, against 16 where eight lanes share 128 bytes (64 rows on 4,096 x 4,096 straight to registers: 21.2 us
// against 11.4).  Rows are swizzled by 16-byte pieces so that a fragment's reads spread over the banks.  Short n: the parts of k leave fp32
// sums in the workspace and a second launch adds them in their order.
// Measured (bf16, weights from HBM, us; library -> this, 64 rows / 16 rows): n 28,672 k 4,096: 56.0 -> 51.2 (4.6 TB/s) / 56.1 -> 46.0;
// 22,016 x 4,096: 50.2 -> 36.4 / 53.0 -> 35.1; 4,096 x 14,336: 37.5 -> 28.7 / 26.3 -> 25.0; 4,096 x 4,096: 13.9 -> 12.2 / 11.9 -> 11.0;
// 1,024 x 4,096: 17.8 -> 9.4; 8,192 x 8,192: 34.3 -> 31.2 / 29.8 -> 28.8 (36.5 with all workgroups beginning at the same stage).  Tiles of
// 112 rows on 28,672 (one workgroup to a compute unit): 50.6.
#include "ops/ops_common.hpp"
#include "ops/vec8.hpp"

namespace hipops {

namespace {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t uint2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

constexpr int kStageBytes = 128;  // of a row in a stage: 64 elements of k

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

typedef __attribute__((address_space(3))) uint8_t lds_byte;
// 16 bytes per lane from global memory to LDS: lane l's land at lds_base + 16 l.  Inline assembly, because the compiler waits
// for the intrinsic form at every access to LDS; waited for by hand.
__device__ __forceinline__ void load_to_lds_16(const char* base, uint32_t lane_offset, lds_byte* lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(lane_offset), "s"(base), "s"((uint32_t)(uintptr_t)lds_base)
                 : "memory", "m0");
}
// everything but the kKeep most recent loads of this wavefront has landed, for every wavefront of the workgroup
template <int kKeep>
__device__ __forceinline__ void barrier_keeping() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070 | (kKeep & 15) | ((kKeep >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

struct MidRowsParams {
    const uint16_t* a;  // [m, k]
    const uint16_t* b;  // [n, k]
    void* c;            // [m, n] of the operands' type or fp32; sums of a part of k: [parts][m][n] fp32
    int m, n;
    int64_t k;
    int tiles, parts, c_is_f32;
};

template <bool kBf16, int kM, int kWaves, int kRing>
__global__ __launch_bounds__(64 * kWaves) void matmul_mid_rows_kernel(MidRowsParams p) {
    constexpr int kTileN = 16 * kWaves, kRows = kTileN + 16 * kM, kSlot = kRows * kStageBytes;
    constexpr int kXLoads = (2 * kM + kWaves - 1) / kWaves, kLoads = 2 + kXLoads;  // loads of a wavefront for a stage, eight rows each
    __shared__ __attribute__((aligned(128))) uint8_t lds[kRing * kSlot];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, row = lane & 15, quarter = lane >> 4;
    const int tile = (int)blockIdx.x % p.tiles, part = (int)blockIdx.x / p.tiles;
    const int stages = (int)(p.k / 64);
    const int first = (int)((int64_t)stages * part / p.parts), count = (int)((int64_t)stages * (part + 1) / p.parts) - first;
    // lane l loads piece (l % 8) ^ (row % 8) of row l / 8, so that the pieces a fragment reads lie on different banks
    const int lrow = lane >> 3, piece = (lane & 7) ^ lrow;
    // workgroups begin at different stages of their part: rows whose distance is a power of two would have all of them wait for the same
    // memory channels
    int stage = (int)((uint32_t)tile * 37u % (uint32_t)max(count, 1));
    const char* const wbase = (const char*)(p.b + (int64_t)(kTileN * tile) * p.k + 64 * (int64_t)first);
    const char* const xbase = (const char*)(p.a + 64 * (int64_t)first);
    uint32_t w[2], x[kXLoads];
    int xrow[kXLoads];
#pragma unroll
    for (int i = 0; i < 2; i++) w[i] = (uint32_t)min(16 * wave + 8 * i + lrow, p.n - 1 - kTileN * tile) * (uint32_t)(2 * p.k) + 16 * piece;
#pragma unroll
    for (int i = 0; i < kXLoads; i++) {
        xrow[i] = 8 * ((kXLoads * wave + i) % (2 * kM));  // (some twice)
        x[i] = (uint32_t)min(xrow[i] + lrow, p.m - 1) * (uint32_t)(2 * p.k) + 16 * piece;
    }
    lds_byte* const base = (lds_byte*)lds;
    const auto load = [&](int slot) __attribute__((always_inline)) {
        const int64_t at = (int64_t)stage * kStageBytes;
#pragma unroll
        for (int i = 0; i < 2; i++) load_to_lds_16(wbase + at, w[i], base + slot * kSlot + (16 * wave + 8 * i) * kStageBytes);
#pragma unroll
        for (int i = 0; i < kXLoads; i++) load_to_lds_16(xbase + at, x[i], base + slot * kSlot + (kTileN + xrow[i]) * kStageBytes);
        stage = stage + 1 == count ? 0 : stage + 1;
    };
    float4_t acc[kM];
#pragma unroll
    for (int i = 0; i < kM; i++) acc[i] = (float4_t){0.f, 0.f, 0.f, 0.f};
    const int at0 = 16 * (quarter ^ (row & 7)), at1 = 16 * ((quarter + 4) ^ (row & 7));
    const auto multiply = [&](int slot) __attribute__((always_inline)) {
        const uint8_t* const s = lds + slot * kSlot + row * kStageBytes;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint4_t wf = *(const uint4_t*)(s + 16 * wave * kStageBytes + (j ? at1 : at0));
#pragma unroll
            for (int i = 0; i < kM; i++) acc[i] = mma<kBf16>(wf, *(const uint4_t*)(s + (kTileN + 16 * i) * kStageBytes + (j ? at1 : at0)), acc[i]);
        }
    };
    for (int i = 0; i < kRing - 1 && i < count; i++) load(i);
    int slot = 0, fill = kRing - 1;
    for (int i = 0; i < count; i++) {
        if (i + kRing - 1 <= count)
            barrier_keeping<(kRing - 2) * kLoads>();  // kRing - 1 stages are on their way: the first is there
        else
            barrier_keeping<0>();
        if (i + kRing - 1 < count) load(fill);  // (into the slot that every wavefront left before the barrier)
        multiply(slot);
        slot = slot + 1 == kRing ? 0 : slot + 1;
        fill = fill + 1 == kRing ? 0 : fill + 1;
    }
    // register r: weight row 4 quarter + r of the wavefront's 16, activation row lane % 16
    const int at = kTileN * tile + 16 * wave + 4 * quarter;  // (n is a multiple of 4)
    if (at >= p.n) return;
#pragma unroll
    for (int i = 0; i < kM; i++) {
        const int out_row = 16 * i + row;
        if (out_row >= p.m) break;
        const int64_t o = ((int64_t)part * p.m + out_row) * p.n + at;
        if (p.parts > 1 || p.c_is_f32)
            *(float4_t*)((float*)p.c + o) = acc[i];
        else
            *(uint2_t*)((uint16_t*)p.c + o) = (uint2_t){cvt2<kBf16>(acc[i][0], acc[i][1]), cvt2<kBf16>(acc[i][2], acc[i][3])};
    }
}

// The parts' sums, in their order; four elements a lane.
template <bool kBf16>
__global__ __launch_bounds__(256) void matmul_sum_parts_kernel(const float* sums, void* c, int64_t count, int parts, int c_is_f32) {
    const int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
    if (i >= count) return;
    float4_t sum = *(const float4_t*)(sums + i);
#pragma unroll 4
    for (int p = 1; p < parts; p++) sum += *(const float4_t*)(sums + p * count + i);
    if (c_is_f32)
        *(float4_t*)((float*)c + i) = sum;
    else
        *(uint2_t*)((uint16_t*)c + i) = (uint2_t){cvt2<kBf16>(sum[0], sum[1]), cvt2<kBf16>(sum[2], sum[3])};
}

struct Split {
    int waves, parts;
};
// Wavefronts to a workgroup and parts of k, by the bytes that the busiest compute unit moves: its share of the weights and, with parts, the
// chip's traffic of their sums.  A part is five stages or more (64 rows: 1,024 x 4,096 in 16 / 12 parts 11.2 / 10.5 us; 2,048 x 2,048 in
// 8 / 6 9.4 / 8.9), four wavefronts unless six deal the rows out better (22,016 x 4,096: 45.8 -> 39.6; 6,144 x 4,096: 17.0 -> 15.3).
Split split_of(int64_t m, int64_t n, int64_t k, size_t workspace_bytes) {
    constexpr int64_t kUnits = 256;
    Split best{4, 1};
    int64_t least = INT64_MAX;
    for (int waves = 4; waves <= 6; waves += 2) {
        const int64_t tiles = (n + 16 * waves - 1) / (16 * waves);
        for (int64_t parts = 1; parts <= 16 && (parts == 1 || (parts * 5 <= k / 64 && parts * tiles <= 2 * kUnits)); parts++) {
            if (parts > 1 && (size_t)(parts * m * n * 4) > workspace_bytes) break;
            const int64_t cost = (tiles * parts + kUnits - 1) / kUnits * (16 * waves) * (2 * k / parts) + (parts > 1 ? parts * m * n * 8 / kUnits : 0);
            if (cost < least) least = cost, best = {waves, (int)parts};
        }
    }
    return best;
}

template <bool kBf16, int kM>
void launch(const MidRowsParams& p, int waves, hipStream_t stream) {
    const dim3 grid((unsigned)(p.tiles * p.parts));
    constexpr int kRing4 = kM == 1 ? 5 : 4, kRing6 = kM == 4 ? 4 : 5;  // (two workgroups to a compute unit, or three)
    if (waves == 4)
        hipLaunchKernelGGL((matmul_mid_rows_kernel<kBf16, kM, 4, kRing4>), grid, dim3(256), 0, stream, p);
    else
        hipLaunchKernelGGL((matmul_mid_rows_kernel<kBf16, kM, 6, kRing6>), grid, dim3(384), 0, stream, p);
}

template <bool kBf16>
void launch(const MidRowsParams& p, int waves, hipStream_t stream) {
    if (p.m <= 16)
        launch<kBf16, 1>(p, waves, stream);
    else if (p.m <= 32)
        launch<kBf16, 2>(p, waves, stream);
    else
        launch<kBf16, 4>(p, waves, stream);
}

}  // namespace

// 16-bit operands, one matrix, the weights' rows along k in whole stages (and 96 rows within 32 bits of offset), 16-byte
// aligned rows.  The sums of the parts need a workspace; without one k stays whole.  The largest weights are the library's
// (128,256 x 4,096 with 7 / 16 / 64 rows: 180 / 191 / 202 us there, 186 / 188 / 206 here).
bool matmul_mid_rows_supported(const hipops_matmul_desc* d, const void* a, const void* b, const void* c) {
    const auto aligned16 = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
    return (d->ab_dtype == HIPATTN_F16 || d->ab_dtype == HIPATTN_BF16) && d->batch == 1 && !d->transpose_a && d->transpose_b && d->m > 6 && d->m <= 64 &&
           d->n % 4 == 0 && d->k % 64 == 0 && d->k < (1 << 24) && d->n * d->k <= (1 << 28) && aligned16(a) && aligned16(b) && aligned16(c);
}

hipattn_status matmul_mid_rows(const hipops_matmul_desc* d, const void* a, const void* b, void* c, void* workspace, size_t workspace_bytes,
                               hipStream_t stream) {
    const Split split = split_of(d->m, d->n, d->k, workspace ? workspace_bytes : 0);
    const bool bf16 = d->ab_dtype == HIPATTN_BF16;
    const int c_is_f32 = d->c_dtype == HIPATTN_F32 ? 1 : 0, rows = 16 * split.waves;
    const MidRowsParams p{(const uint16_t*)a, (const uint16_t*)b, split.parts > 1 ? workspace : c, (int)d->m, (int)d->n, d->k,
                          (int)((d->n + rows - 1) / rows), split.parts, c_is_f32};
    if (bf16)
        launch<true>(p, split.waves, stream);
    else
        launch<false>(p, split.waves, stream);
    if (split.parts > 1) {
        const int64_t count = d->m * d->n;
        const dim3 grid((unsigned)((count / 4 + 255) / 256));
        const auto kernel = bf16 ? matmul_sum_parts_kernel<true> : matmul_sum_parts_kernel<false>;
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, (const float*)workspace, c, count, split.parts, c_is_f32);
    }
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return fail(HIPATTN_HIP_ERROR, "matmul: %s", hipGetErrorString(e));
    return HIPATTN_OK;
}

}  // namespace hipops
