// Products of few activation rows with a weight matrix stored [n, k] -- the projections of a decode step of a serving batch -- on
// v_mfma_f32_16x16x32 with fp32 accumulation, instead of the library's kernels: of 7 to 64 rows by themselves, of 1 to 64 with what follows
// them (projection()).
//
// What bounds it: the weights, read once from HBM.  A workgroup takes 64, 96 or 128 weight rows and a part
// of k; weights and activations come to LDS 64 elements of k at a time (global_load_lds, a ring of kRing stages, one barrier to a stage),
// because the matrix operands as they stand are not what a compute unit loads well: sixteen lanes in sixteen rows take
// 64 clocks to an instruction, against 16 where eight lanes share 128 bytes (64 rows on 4,096 x 4,096 straight to registers: 21.2 us
// against 11.4).  Rows are swizzled by 16-byte pieces so that a fragment's reads spread over the banks.  Short n: the parts of k leave fp32
// sums in the workspace and a second launch adds them in their order.
// Measured (bf16, weights from HBM, us; library -> this, 64 rows / 16 rows): n 28,672 k 4,096: 52.7 -> 43.6 (5.4 TB/s) / 56.1 -> 46.0;
// 22,016 x 4,096: 50.2 -> 37.1 / 53.0 -> 35.1; 4,096 x 14,336: 37.5 -> 28.7 / 26.3 -> 25.0; 4,096 x 4,096: 13.9 -> 12.2 / 11.9 -> 11.0;
// 1,024 x 4,096: 17.8 -> 9.4; 8,192 x 8,192: 34.3 -> 31.2 / 29.8 -> 28.8 (36.5 with all workgroups beginning at the same stage).
// Two tiles of 16 weight rows to a wavefront read its activations from LDS half as often: 50.2 -> 43.4 at 28,672 x 4,096, 64 rows.
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

constexpr int kMaxWeights = 3;

struct MidRowsParams {
    const uint16_t* a;               // [m, k]
    const uint16_t* b[kMaxWeights];  // [n[i], k]
    void* c[kMaxWeights];            // [m, n[i]] of the operands' type or fp32; not written where there are sums
    float* sums;                     // null, or the parts' sums: [parts][m][sum of n] fp32
    int n[kMaxWeights];
    int begin[kMaxWeights];          // the first tile of weights i
    int offset[kMaxWeights];         // their first column in a row of sums
    int m, columns, tiles, parts, c_is_f32;
    int activation, gate_first;      // kGlu
    int64_t k;
};

// kGlu: the weight rows are the two halves of a gated MLP; a wavefront's 16 are eight of the gate's and the same eight of the other half,
// c is [m, n / 2].
template <bool kBf16, bool kGlu, int kM, int kWaves, int kN, int kRing>
__global__ __launch_bounds__(64 * kWaves) void matmul_mid_rows_kernel(MidRowsParams p) {
    constexpr int kTileN = 16 * kN * kWaves, kRows = kTileN + 16 * kM, kSlot = kRows * kStageBytes;
    constexpr int kXLoads = (2 * kM + kWaves - 1) / kWaves, kLoads = 2 * kN + kXLoads;  // loads of a wavefront for a stage, eight rows each
    __shared__ __attribute__((aligned(128))) uint8_t lds[kRing * kSlot];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, row = lane & 15, quarter = lane >> 4;
    const int tile_of_all = (int)blockIdx.x % p.tiles, part = (int)blockIdx.x / p.tiles;
    const int which = (tile_of_all >= p.begin[1]) + (tile_of_all >= p.begin[2]);  // (absent weights begin behind the last tile)
    const int tile = tile_of_all - p.begin[which], n = p.n[which];
    const int stages = (int)(p.k / 64);
    const int first = (int)((int64_t)stages * part / p.parts), count = (int)((int64_t)stages * (part + 1) / p.parts) - first;
    // lane l loads piece (l % 8) ^ (row % 8) of row l / 8, so that the pieces a fragment reads lie on different banks
    const int lrow = lane >> 3, piece = (lane & 7) ^ lrow;
    // workgroups begin at different stages of their part: rows whose distance is a power of two would have all of them wait for the same
    // memory channels
    int stage = (int)((uint32_t)tile_of_all * 37u % (uint32_t)max(count, 1));
    const char* const wbase = (const char*)(p.b[which] + 64 * (int64_t)first);
    const char* const xbase = (const char*)(p.a + 64 * (int64_t)first);
    uint32_t w[2 * kN], x[kXLoads];
    int xrow[kXLoads];
#pragma unroll
    for (int i = 0; i < 2 * kN; i++) {
        const int row0 = kTileN * tile + 16 * (kN * wave + i / 2);
        int r = min(row0 + 8 * (i & 1) + lrow, n - 1);
        if constexpr (kGlu) r = min(row0 / 2 + lrow, n / 2 - 1) + (p.gate_first ? i & 1 : 1 - (i & 1)) * (n / 2);
        w[i] = (uint32_t)r * (uint32_t)(2 * p.k) + 16 * piece;
    }
#pragma unroll
    for (int i = 0; i < kXLoads; i++) {
        xrow[i] = 8 * ((kXLoads * wave + i) % (2 * kM));  // (some twice)
        x[i] = (uint32_t)min(xrow[i] + lrow, p.m - 1) * (uint32_t)(2 * p.k) + 16 * piece;
    }
    lds_byte* const base = (lds_byte*)lds;
    const auto load = [&](int slot) __attribute__((always_inline)) {
        const int64_t at = (int64_t)stage * kStageBytes;
#pragma unroll
        for (int i = 0; i < 2 * kN; i++) load_to_lds_16(wbase + at, w[i], base + slot * kSlot + (16 * kN * wave + 8 * i) * kStageBytes);
#pragma unroll
        for (int i = 0; i < kXLoads; i++) load_to_lds_16(xbase + at, x[i], base + slot * kSlot + (kTileN + xrow[i]) * kStageBytes);
        stage = stage + 1 == count ? 0 : stage + 1;
    };
    float4_t acc[kN][kM];
#pragma unroll
    for (int t = 0; t < kN; t++)
#pragma unroll
        for (int i = 0; i < kM; i++) acc[t][i] = (float4_t){0.f, 0.f, 0.f, 0.f};
    const int at0 = 16 * (quarter ^ (row & 7)), at1 = 16 * ((quarter + 4) ^ (row & 7));
    const auto multiply = [&](int slot) __attribute__((always_inline)) {
        const uint8_t* const s = lds + slot * kSlot + row * kStageBytes;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            uint4_t wf[kN];
#pragma unroll
            for (int t = 0; t < kN; t++) wf[t] = *(const uint4_t*)(s + 16 * (kN * wave + t) * kStageBytes + (j ? at1 : at0));
#pragma unroll
            for (int i = 0; i < kM; i++) {
                const uint4_t xf = *(const uint4_t*)(s + (kTileN + 16 * i) * kStageBytes + (j ? at1 : at0));
#pragma unroll
                for (int t = 0; t < kN; t++) acc[t][i] = mma<kBf16>(wf[t], xf, acc[t][i]);
            }
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
    // register r: weight row 4 quarter + r of the 16, activation row lane % 16
#pragma unroll
    for (int t = 0; t < kN; t++) {
        const int row0 = kTileN * tile + 16 * (kN * wave + t);
        if constexpr (kGlu) {
            const int at = row0 / 2 + 4 * quarter;  // (of quarters 0 and 1; n / 2 is a multiple of 4)
#pragma unroll
            for (int i = 0; i < kM; i++) {
                float4_t other, o;
#pragma unroll
                for (int r = 0; r < 4; r++) other[r] = __shfl_xor(acc[t][i][r], 32);
                const int out_row = 16 * i + row;
                if (quarter > 1 || at >= n / 2 || out_row >= p.m) continue;
#pragma unroll
                for (int r = 0; r < 4; r++) o[r] = activate(acc[t][i][r], p.activation, 1.0f) * other[r];
                *(uint2_t*)((uint16_t*)p.c[0] + (int64_t)out_row * (n / 2) + at) = (uint2_t){cvt2<kBf16>(o[0], o[1]), cvt2<kBf16>(o[2], o[3])};
            }
            continue;
        }
        const int at = row0 + 4 * quarter;  // (n is a multiple of 4)
        if (at >= n) continue;
#pragma unroll
        for (int i = 0; i < kM; i++) {
            const int out_row = 16 * i + row;
            if (out_row >= p.m) break;
            const int64_t o = (int64_t)out_row * n + at;
            if (p.sums != nullptr)
                *(float4_t*)(p.sums + ((int64_t)part * p.m + out_row) * p.columns + p.offset[which] + at) = acc[t][i];
            else if (p.c_is_f32)
                *(float4_t*)((float*)p.c[which] + o) = acc[t][i];
            else
                *(uint2_t*)((uint16_t*)p.c[which] + o) = (uint2_t){cvt2<kBf16>(acc[t][i][0], acc[t][i][1]), cvt2<kBf16>(acc[t][i][2], acc[t][i][3])};
        }
    }
}

__device__ __forceinline__ float4_t add_parts(const float* sums, int64_t part_stride, int parts) {
    float4_t sum = *(const float4_t*)sums;
#pragma unroll 4
    for (int p = 1; p < parts; p++) sum += *(const float4_t*)(sums + p * part_stride);
    return sum;
}

// The parts' sums, in their order; four elements a lane.
template <bool kBf16>
__global__ __launch_bounds__(256) void matmul_sum_parts_kernel(const float* sums, void* c, int64_t count, int parts, int c_is_f32) {
    const int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
    if (i >= count) return;
    const float4_t sum = add_parts(sums + i, count, parts);
    if (c_is_f32)
        *(float4_t*)((float*)c + i) = sum;
    else
        *(uint2_t*)((uint16_t*)c + i) = (uint2_t){cvt2<kBf16>(sum[0], sum[1]), cvt2<kBf16>(sum[2], sum[3])};
}

struct FinishParams {
    const float* sums;
    void* out[kMaxWeights];
    int n[kMaxWeights], offset[kMaxWeights];
    int m, columns, parts, dtype;
    int rotated, head_size;  // rotated: a bit for each output
    const void *cos, *sin;
    const int32_t* positions;
    int64_t table_row_stride;
    int table_dtype, gamma_dtype;
    const void *residual, *gamma;
    void* normalised;
    float eps;
    const void* product;  // instead of sums, where another kernel has finished it
};

// What follows the products, on the parts' sums: a rotary embedding of some outputs, or a residual; eight elements a lane, of a rotated
// head four of each half.  Replaces a launch for each, which is most of what these cost (4 to 5 us each for a serving batch).
__global__ __launch_bounds__(256) void projection_finish_kernel(FinishParams p) {
    const int item = (int)blockIdx.x * 256 + threadIdx.x, row = (int)blockIdx.y;
    if (8 * item >= p.columns) return;
    const int which = (8 * item >= p.offset[1]) + (8 * item >= p.offset[2]);
    const int local = item - p.offset[which] / 8;
    const bool rotate = (p.rotated >> which) & 1;
    int c0 = 8 * local, c1 = c0 + 4, i = 0;
    const int half = p.head_size / 2;
    if (rotate) {
        const int head = local / (p.head_size / 8);
        i = 4 * (local - head * (p.head_size / 8));
        c0 = head * p.head_size + i, c1 = c0 + half;
    }
    const int64_t stride = (int64_t)p.m * p.columns;
    const float* const s = p.sums + (int64_t)row * p.columns + p.offset[which];
    const float4_t lo = add_parts(s + c0, stride, p.parts), hi = add_parts(s + c1, stride, p.parts);
    float4_t ol = lo, oh = hi;
    const int64_t base = (int64_t)row * p.n[which];
    if (rotate) {
        const int64_t tb = (p.positions ? (int64_t)p.positions[row] : row) * p.table_row_stride + i;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            ol[k] = lo[k] * load_scalar(p.cos, tb + k, p.table_dtype) - hi[k] * load_scalar(p.sin, tb + k, p.table_dtype);
            oh[k] = hi[k] * load_scalar(p.cos, tb + half + k, p.table_dtype) + lo[k] * load_scalar(p.sin, tb + half + k, p.table_dtype);
        }
    } else if (p.residual != nullptr) {
        const Float8 r = load8(p.residual, base + c0, p.dtype);
#pragma unroll
        for (int k = 0; k < 4; k++) ol[k] += r.v[k], oh[k] += r.v[4 + k];
    }
    const auto store = [&](int64_t at, const float4_t& v) {
        *(uint2_t*)((uint16_t*)p.out[which] + at) = p.dtype == HIPATTN_BF16 ? (uint2_t){cvt2<true>(v[0], v[1]), cvt2<true>(v[2], v[3])}
                                                                            : (uint2_t){cvt2<false>(v[0], v[1]), cvt2<false>(v[2], v[3])};
    };
    store(base + c0, ol);
    store(base + c1, oh);
}

constexpr int kNormThreads = 512, kNormKeep = 4;  // chunks of eight elements that a lane keeps: rows of up to 16,384

// The residual added to the parts' sums, or to a finished product, and the RMS norm of the rounded result; a workgroup to a row.  Bounded by
// HBM where rows are many: two tensors read and two written once (us as two operators -> here: 100 rows of 4,096 7.5 -> 3.8, 2,224 20.6 -> 14.4,
// 8,000 54.5 -> 38.5 (5.4 TB/s); 6,000 of 2,048 27.1 -> 17.1, 30.3 with workgroups of 512 lanes for any row).
// kKeep: chunks to a lane; 1 for rows of up to 4,096, whose workgroups are then as wide as the row.
template <int kKeep>
__global__ __launch_bounds__(kNormThreads) void projection_norm_kernel(FinishParams p) {
    __shared__ float partial[kNormThreads / 64];
    const int64_t base = (int64_t)blockIdx.x * p.columns, stride = (int64_t)p.m * p.columns;
    const int chunks = p.columns / 8;
    Float8 keep[kKeep], gamma[kKeep];
    float sq = 0.f;
#pragma unroll
    for (int c = 0; c < kKeep; c++) {
        const int ch = threadIdx.x + c * (int)blockDim.x;
        if (ch < chunks) {
            gamma[c] = load8(p.gamma, 8 * ch, p.gamma_dtype);
            Float8 r = load8(p.residual, base + 8 * ch, p.dtype);
            if (p.product != nullptr) {
                const Float8 x = load8(p.product, base + 8 * ch, p.dtype);
#pragma unroll
                for (int k = 0; k < 8; k++) r.v[k] += x.v[k];
            } else {
                const float4_t lo = add_parts(p.sums + base + 8 * ch, stride, p.parts), hi = add_parts(p.sums + base + 8 * ch + 4, stride, p.parts);
#pragma unroll
                for (int k = 0; k < 4; k++) r.v[k] += lo[k], r.v[4 + k] += hi[k];
            }
            store8(p.out[0], base + 8 * ch, p.dtype, r);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                keep[c].v[k] = p.dtype == HIPATTN_BF16 ? (float)(__bf16)r.v[k] : (float)(_Float16)r.v[k];
                sq = fmaf(keep[c].v[k], keep[c].v[k], sq);
            }
        }
    }
    sq = wave_sum(sq);
    if ((threadIdx.x & 63) == 0) partial[threadIdx.x / 64] = sq;
    __syncthreads();
    sq = 0.f;
#pragma unroll
    for (int w = 0; w < kNormThreads / 64; w++) sq += w < (int)blockDim.x / 64 ? partial[w] : 0.f;
    const float inv = 1.0f / sqrtf(sq / (float)p.columns + p.eps);
#pragma unroll
    for (int c = 0; c < kKeep; c++) {
        const int ch = threadIdx.x + c * (int)blockDim.x;
        if (ch < chunks) {
            Float8 o;
#pragma unroll
            for (int k = 0; k < 8; k++) o.v[k] = (keep[c].v[k] * inv) * gamma[c].v[k];
            store8(p.normalised, base + 8 * ch, p.dtype, o);
        }
    }
}

constexpr int64_t kMaxParts = 16;
struct Split {
    int rows, parts;
};
// Weight rows to a workgroup (64, 96 or 128) and parts of k, by the bytes that the busiest compute unit moves: its weights, a quarter of its
// activations (they come from the L2) and, with parts, twice the chip's traffic of their sums, which the second launch waits for.  A part is
// five stages or more.  (us without the second launch, 64 rows, 64 / 96 / 128 weight rows at their best parts: 28,672 x 4,096 50.2 / 53 / 43.4;
// 22,016 x 4,096 42.2 / 35.8 / 38.4; 6,144 x 4,096 14.6 / 13.0 / 13.5; 4,096 x 4,096 9.6 / 10.8 / 10.5; 4,096 x 14,336 25.3 / 27 / 25.5.)
// 128 rows for more than 16 activation rows only: with fewer the activations are no burden.
Split split_of(int64_t m, const int64_t* n, int count, int64_t k, size_t workspace_bytes, bool whole_k) {
    constexpr int64_t kUnits = 256;
    Split best{64, 1};
    int64_t least = INT64_MAX, columns = 0;
    for (int i = 0; i < count; i++) columns += n[i];
    const int64_t activations = m <= 16 ? 16 : m <= 32 ? 32 : 64;
    for (int rows = 64; rows <= (m > 16 ? 128 : 96); rows += 32) {
        int64_t tiles = 0;
        for (int i = 0; i < count; i++) tiles += (n[i] + rows - 1) / rows;
        for (int64_t parts = 1; parts <= kMaxParts && (parts == 1 || (!whole_k && parts * 5 <= k / 64 && parts * tiles <= 2 * kUnits)); parts++) {
            if (parts > 1 && (size_t)(parts * m * columns * 4) > workspace_bytes) break;
            const int64_t cost =
                (tiles * parts + kUnits - 1) / kUnits * (rows + activations / 4) * (2 * k / parts) + (parts > 1 ? parts * m * columns * 16 / kUnits : 0);
            if (cost < least) least = cost, best = {rows, (int)parts};
        }
    }
    return best;
}

void launch_norm(const FinishParams& f, hipStream_t stream) {
    const int chunks = f.columns / 8;
    if (chunks <= kNormThreads)
        hipLaunchKernelGGL(projection_norm_kernel<1>, dim3((unsigned)f.m), dim3((unsigned)((chunks + 63) / 64 * 64)), 0, stream, f);
    else
        hipLaunchKernelGGL(projection_norm_kernel<kNormKeep>, dim3((unsigned)f.m), dim3(kNormThreads), 0, stream, f);
}

// (rings: two workgroups to a compute unit, or three)
template <bool kBf16, bool kGlu, int kM>
void launch(const MidRowsParams& p, int rows, hipStream_t stream) {
    const dim3 grid((unsigned)(p.tiles * p.parts));
    if constexpr (kM > 1) {
        if (rows == 128) {
            hipLaunchKernelGGL((matmul_mid_rows_kernel<kBf16, kGlu, kM, 4, 2, kM == 4 ? 3 : 4>), grid, dim3(256), 0, stream, p);
            return;
        }
    }
    if (rows == 64)
        hipLaunchKernelGGL((matmul_mid_rows_kernel<kBf16, kGlu, kM, 4, 1, kM == 1 ? 5 : 4>), grid, dim3(256), 0, stream, p);
    else
        hipLaunchKernelGGL((matmul_mid_rows_kernel<kBf16, kGlu, kM, 6, 1, kM == 4 ? 4 : 5>), grid, dim3(384), 0, stream, p);
}

template <bool kBf16, bool kGlu>
void launch(const MidRowsParams& p, int rows, hipStream_t stream) {
    if (p.m <= 16)
        launch<kBf16, kGlu, 1>(p, rows, stream);
    else if (p.m <= 32)
        launch<kBf16, kGlu, 2>(p, rows, stream);
    else
        launch<kBf16, kGlu, 4>(p, rows, stream);
}

// the products of one input with `count` weights, in tiles of split.rows
MidRowsParams params_of(const void* a, const void* const* b, void* const* c, const int64_t* n, int count, int64_t m, int64_t k, const Split& split,
                        float* sums) {
    MidRowsParams p{};
    p.a = (const uint16_t*)a, p.sums = sums, p.m = (int)m, p.k = k, p.parts = split.parts;
    for (int i = 0; i < kMaxWeights; i++) {
        p.begin[i] = INT32_MAX;
        if (i >= count) continue;
        p.b[i] = (const uint16_t*)b[i], p.c[i] = c[i], p.n[i] = (int)n[i];
        p.begin[i] = p.tiles, p.offset[i] = p.columns;
        p.tiles += (int)((n[i] + split.rows - 1) / split.rows), p.columns += (int)n[i];
    }
    return p;
}

bool aligned16(const void* x) { return ((uintptr_t)x & 15) == 0; }
bool overlap(const void* a, int64_t a_bytes, const void* b, int64_t b_bytes) {
    return (uintptr_t)a < (uintptr_t)b + (uintptr_t)b_bytes && (uintptr_t)b < (uintptr_t)a + (uintptr_t)a_bytes;
}
// Operator by operator the sum of all rows is there before the norm of any is written; here another row's workgroup may still be reading.  (The
// residual's own place is fine: what a lane writes there it has read.)
bool norm_over_inputs(const void* residual, const void* gamma, int gamma_dtype, const void* out, const void* normalised, int64_t rows, int64_t n) {
    const int64_t bytes = 2 * rows * n, gamma_bytes = n * (gamma_dtype == HIPATTN_F32 ? 4 : 2);
    return (normalised != residual && overlap(normalised, bytes, residual, bytes)) || overlap(out, bytes, gamma, gamma_bytes);
}

// Where the library's kernels are the faster ones (us, library / this).
bool library_is_faster(int64_t m, int64_t n, int64_t k, size_t workspace_bytes) {
    // A workspace too small for the parts of k (or none): a workgroup's chain of k, where the workgroups are fewer than two thirds of the compute
    // units (no workspace; 16 rows, 4,096 x 2,048 11.0 / 8.9, x 2,560 11.4 / 12.0, 8,192 x 4,096 16.1 / 17.5, 9,216 x 4,096 23.8 / 18.1, 16 x 8,192 11.0 / 26.1;
    // 32 rows, 512 x 2,048 11.1 / 9.7, x 2,560 11.3 / 11.5, x 3,072 10.9 / 13.4; 64 rows, 512 x 1,536 11.1 / 9.8, x 2,048 11.1 / 12.2, 4,096 x 4,096 14.0 / 22.1,
    // 11,008 x 4,096 27.0 / 25.0).
    const int64_t longest = m <= 32 ? 2048 : 1536;
    if (k > longest && n < 172 * 64 && workspace_bytes < (size_t)(kMaxParts * m * n * 4)) {
        const int64_t parts = split_of(m, &n, 1, k, workspace_bytes, false).parts;
        if (n * parts < 172 * 64 && k / parts > longest && parts < split_of(m, &n, 1, k, SIZE_MAX, false).parts) return true;
    }
    // Up to 16 rows on some middling weights (16 rows: 2,560 x 5,120 10.6 / 10.1, 2,816 x 5,120 10.6 / 11.2, 3,328 x 5,120 10.8 / 11.8, x 9,216 15.9 / 15.9,
    // 4,096 x 8,192 15.8 / 17.6, x 10,240 19.5 / 19.3, 4,608 x 8,192 22.4 / 18.7; 24 rows: 3,328 x 5,120 12.9 / 12.2) and, to 32 rows from n = 7,168 on, on short k (16 rows:
    // 5,632 x 3,072 11.2 / 11.6, 6,144 x 3,072 10.9 / 11.9, 8,192 x 4,096 15.7 / 17.8, x 6,144 23.7 / 21.3, 9,216 x 4,096 23.6 / 20.4; 32 rows: 6,144 x 4,096 14.8 / 14.3,
    // 8,192 x 4,096 16.2 / 18.2).
    if (m <= 16 && n >= 2816 && n <= 4096 && k >= 5120 && k <= 9216) return true;
    return m <= (n < 7168 ? 16 : 32) && n >= 6144 && n <= 8192 && k >= 3072 && k <= 5120;
}

bool sizes_supported(int dtype, int64_t n, int64_t k) {
    return (dtype == HIPATTN_F16 || dtype == HIPATTN_BF16) && k % 64 == 0 && k < (1 << 24) && n * k <= (1 << 28);
}

}  // namespace

// 16-bit operands, one matrix, the weights' rows along k in whole stages (and all of them within 32 bits of offset), 16-byte
// aligned rows.  The sums of the parts need a workspace; without one k stays whole.  The largest weights are the library's
// (128,256 x 4,096 with 7 / 16 / 64 rows: 180 / 191 / 202 us there, 186 / 188 / 206 here), and so is what library_is_faster names.
bool matmul_mid_rows_supported(const hipops_matmul_desc* d, const void* a, const void* b, const void* c, size_t workspace_bytes) {
    return sizes_supported(d->ab_dtype, d->n, d->k) && d->batch == 1 && !d->transpose_a && d->transpose_b && d->m > 6 && d->m <= 64 && d->n % 4 == 0 &&
           aligned16(a) && aligned16(b) && aligned16(c) && !library_is_faster(d->m, d->n, d->k, workspace_bytes);
}

hipattn_status matmul_mid_rows(const hipops_matmul_desc* d, const void* a, const void* b, void* c, void* workspace, size_t workspace_bytes,
                               hipStream_t stream) {
    const Split split = split_of(d->m, &d->n, 1, d->k, workspace ? workspace_bytes : 0, false);
    const bool bf16 = d->ab_dtype == HIPATTN_BF16;
    MidRowsParams p = params_of(a, &b, &c, &d->n, 1, d->m, d->k, split, split.parts > 1 ? (float*)workspace : nullptr);
    p.c_is_f32 = d->c_dtype == HIPATTN_F32 ? 1 : 0;
    if (bf16)
        launch<true, false>(p, split.rows, stream);
    else
        launch<false, false>(p, split.rows, stream);
    if (split.parts > 1) {
        const int64_t count = d->m * d->n;
        const dim3 grid((unsigned)((count / 4 + 255) / 256));
        const auto kernel = bf16 ? matmul_sum_parts_kernel<true> : matmul_sum_parts_kernel<false>;
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, p.sums, c, count, split.parts, p.c_is_f32);
    }
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return fail(HIPATTN_HIP_ERROR, "matmul: %s", hipGetErrorString(e));
    return HIPATTN_OK;
}

// Up to 64 rows: one launch for all the products of an input and one for what follows them, where the operators one by one are a
// launch each.  Bounded by the weights, once launches are few: us, 4 / 64 rows of hidden 4,096, 32 / 8 heads of 128, MLP 14,336: q, k, v and
// two rotary embeddings in five to eight launches 33 / 62 -> 15.6 / 20.1; o, residual and norm 18 / 34 -> 13.7 / 16.2; gate|up and SwiGLU
// 47 / 57 -> 42.0 / 46; down and residual 26 / 42 -> 25.8 / 31.8.
// Over the sizes (1 to 64 rows, n 64 to 8,192, k 256 to 16,384, weights from HBM, us in a recorded graph): with a rotary embedding 1.4 to 4 times
// as fast everywhere, with the norm 1.05 to 2 times.  A residual alone is 0.9 to 1.9 times: two launches either way, and up to 8 rows the kernel of few rows
// wins by up to 1.4 us where its wavefronts' k is whole rounds (4 rows: 512 x 1,024 5.8 / 6.6, 3,072 x 3,072 10.4 / 11.1, 4,096 x 8,192 18.1 / 19.3;
// but 4,096 x 7,168 17.9 / 17.0, 5,120 x 8,192 28.1 / 20.9): too little, and of a model's last Add only, for a line of its own.
hipattn_status projection(const hipops_projection_desc* d, const hipops_projection_args* t, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    if (!d || !t) return fail(HIPATTN_INVALID_ARGUMENT, "projection: null descriptor");
    const auto refuse = [](const char* why) { return fail(HIPATTN_UNSUPPORTED, "projection: %s", why); };
    if (d->num_weights < 1 || d->num_weights > kMaxWeights) return refuse("one to three weights");
    if (d->rows < 1 || d->rows > 64) return refuse("1 to 64 rows");
    const bool glu = d->kind == HIPOPS_PROJECTION_GLU, add = d->kind == HIPOPS_PROJECTION_ADD, rope = d->kind == HIPOPS_PROJECTION_ROPE;
    if (!glu && !add && !rope) return fail(HIPATTN_INVALID_ARGUMENT, "projection: kind %d", d->kind);
    if ((glu || add) && d->num_weights != 1) return refuse("several weights go with a rotary embedding only");
    int64_t columns = 0;
    for (int i = 0; i < d->num_weights; i++) {
        if (d->n[i] < 1 || d->n[i] % 8 != 0 || !sizes_supported(d->dtype, d->n[i], d->k) || d->k < 64) return refuse("types or sizes");
        if (!t->weights[i] || !t->outs[i]) return fail(HIPATTN_INVALID_ARGUMENT, "projection: null pointer");
        if (!aligned16(t->weights[i]) || !aligned16(t->outs[i])) return refuse("operands off 16 bytes");
        columns += d->n[i];
    }
    if (!t->x) return fail(HIPATTN_INVALID_ARGUMENT, "projection: null pointer");
    if (!aligned16(t->x)) return refuse("operands off 16 bytes");
    const bool bf16 = d->dtype == HIPATTN_BF16;
    if (glu) {
        if (d->glu_activation < HIPOPS_GLU_SWISH || d->glu_activation > HIPOPS_GLU_GELU_TANH)
            return fail(HIPATTN_INVALID_ARGUMENT, "projection: activation %d", d->glu_activation);
        // k stays whole: where the weights are too few rows for two thirds of the compute units a long one is a chain that the product in parts and
        // the GLU as an operator are faster than (us, one by one / here; 4 rows: 512 x 2,048 7.7 / 9.3, 7,168 x 2,048 13.0 / 12.2; 16 rows: 512 x 2,048 8.9 / 9.1,
        // x 4,096 12.5 / 15.4, x 8,192 11 / 28; 32 rows: 8,192 x 2,048 15.2 / 14.7, x 4,096 20.5 / 23.6; 64 rows: 2,048 x 2,048 12.1 / 14.0, 8,192 x 2,048
        // 16.7 / 16.2, x 8,192 36 / 46; 11,264 x 4,096 28 / 29, 33 with the library's product)
        const bool enough = (d->rows > 8 && d->rows <= 32) || d->n[0] >= (d->rows <= 8 ? 7168 : 4096);
        if (d->n[0] < 172 * 64 && d->k > (enough ? 2048 : 1536)) return refuse("k too long for weights of few rows");
        // (the operators one by one read x before they write over it; here other workgroups may still be reading)
        if (overlap(t->x, 2 * d->rows * d->k, t->outs[0], d->rows * d->n[0])) return refuse("results over the input");
        const Split split = split_of(d->rows, d->n, 1, d->k, 0, true);
        MidRowsParams p = params_of(t->x, t->weights, t->outs, d->n, 1, d->rows, d->k, split, nullptr);
        p.activation = d->glu_activation, p.gate_first = d->glu_gate_first ? 1 : 0;
        if (bf16)
            launch<true, true>(p, split.rows, stream);
        else
            launch<false, true>(p, split.rows, stream);
    } else {
        const auto float_type = [](int x) { return x == HIPATTN_F32 || x == HIPATTN_F16 || x == HIPATTN_BF16; };
        if (add && (!t->residual || (t->gamma == nullptr) != (t->normalised == nullptr))) return fail(HIPATTN_INVALID_ARGUMENT, "projection: null pointer");
        if (add && (!aligned16(t->residual) || !aligned16(t->gamma) || !aligned16(t->normalised))) return refuse("operands off 16 bytes");
        if (t->gamma && (!float_type(d->gamma_dtype) || columns > 8 * kNormThreads * kNormKeep)) return refuse("gamma or row length of the norm");
        if (add && t->gamma && norm_over_inputs(t->residual, t->gamma, d->gamma_dtype, t->outs[0], t->normalised, d->rows, columns)) return refuse("results over an input");
        if (rope && d->rotated_outputs) {
            if (!t->cos || !t->sin) return fail(HIPATTN_INVALID_ARGUMENT, "projection: null pointer");
            if (d->head_size < 8 || d->head_size % 8 != 0 || !float_type(d->table_dtype)) return refuse("head size or table type");
            for (int i = 0; i < d->num_weights; i++)
                if (((d->rotated_outputs >> i) & 1) && d->n[i] % d->head_size != 0) return refuse("rows of no whole heads");
        }
        if (!workspace || !aligned16(workspace) || workspace_bytes < (size_t)(d->rows * columns * 4)) return refuse("no workspace for the sums");
        const Split split = split_of(d->rows, d->n, d->num_weights, d->k, workspace_bytes, false);
        const MidRowsParams p = params_of(t->x, t->weights, t->outs, d->n, d->num_weights, d->rows, d->k, split, (float*)workspace);
        if (bf16)
            launch<true, false>(p, split.rows, stream);
        else
            launch<false, false>(p, split.rows, stream);
        FinishParams f{};
        f.sums = p.sums, f.m = p.m, f.columns = p.columns, f.parts = p.parts, f.dtype = d->dtype;
        for (int i = 0; i < kMaxWeights; i++) {
            f.out[i] = p.c[i], f.n[i] = p.n[i];
            f.offset[i] = i < d->num_weights ? p.offset[i] : INT32_MAX;
        }
        if (add) {
            f.residual = t->residual, f.gamma = t->gamma, f.normalised = t->normalised, f.gamma_dtype = d->gamma_dtype, f.eps = d->eps;
        } else {
            f.rotated = d->rotated_outputs, f.head_size = d->head_size, f.cos = t->cos, f.sin = t->sin, f.positions = t->positions;
            f.table_row_stride = d->table_row_stride, f.table_dtype = d->table_dtype;
        }
        if (f.gamma)
            launch_norm(f, stream);
        else
            hipLaunchKernelGGL(projection_finish_kernel, dim3((unsigned)((columns / 8 + 255) / 256), (unsigned)p.m), dim3(256), 0, stream, f);
    }
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return fail(HIPATTN_HIP_ERROR, "projection: %s", hipGetErrorString(e));
    return HIPATTN_OK;
}

hipattn_status residual_norm(const void* product, const void* residual, const void* gamma, void* out, void* normalised, int64_t rows, int64_t n,
                             float eps, int dtype, int gamma_dtype, hipStream_t stream) {
    const auto refuse = [](const char* why) { return fail(HIPATTN_UNSUPPORTED, "residual_norm: %s", why); };
    if (!product || !residual || !gamma || !out || !normalised) return fail(HIPATTN_INVALID_ARGUMENT, "residual_norm: null pointer");
    if ((dtype != HIPATTN_F16 && dtype != HIPATTN_BF16) || (gamma_dtype != HIPATTN_F32 && gamma_dtype != HIPATTN_F16 && gamma_dtype != HIPATTN_BF16))
        return refuse("types");
    if (rows < 1 || rows > 0x7fffffffLL || n < 8 || n % 8 != 0 || n > 8 * kNormThreads * kNormKeep) return refuse("sizes");
    if (!aligned16(product) || !aligned16(residual) || !aligned16(gamma) || !aligned16(out) || !aligned16(normalised)) return refuse("operands off 16 bytes");
    if (norm_over_inputs(residual, gamma, gamma_dtype, out, normalised, rows, n)) return refuse("results over an input");
    FinishParams f{};
    f.product = product, f.residual = residual, f.gamma = gamma, f.out[0] = out, f.normalised = normalised;
    f.columns = (int)n, f.m = (int)rows, f.dtype = dtype, f.gamma_dtype = gamma_dtype, f.eps = eps;
    launch_norm(f, stream);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return fail(HIPATTN_HIP_ERROR, "residual_norm: %s", hipGetErrorString(e));
    return HIPATTN_OK;
}

}  // namespace hipops
