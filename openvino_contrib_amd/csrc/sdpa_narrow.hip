// Dense attention of 16-bit operands at head sizes 64 and 72 .. 128: both products on v_mfma_f32_32x32x16, laid out
// as in flash_prefill.hip (S^T = K Q^T with the softmax's reference in the accumulator, O^T = V^T P^T).
//
// What bounds it: below 128 a key tile has as many exponentials as at 128 and half to three quarters of
// the matrix work, so the vector ALU is the busier unit (32 x 32 scores: 352 cycles of exp2, sum and conversion
// against 256 of MFMAs at head size 64), and what counts is that it never waits.  So: small workgroups of four
// wavefronts, 32 query rows each, several of them to a compute unit, which find their own phases; a wavefront computes the
// scores of the next 32 keys and the products of the last beside the exponentials of these; no row maximum unless a sum says
// that one is needed.  K and V tiles go straight into LDS, K in three stages (it is read half a tile ahead) and V in two.
// Row sums are taken of the probabilities as they were rounded for the product, so that rounding them moves a row's mean less.
//
// Counters at 16 heads of 4,096, size 64: vector ALU 45 %, matrix cores 40 % of the busy cycles (16 x 16 of 577: 53 %, 36 %), no bank
// conflicts; the rest is a step's own chain (LDS, products, exponentials, check) at two wavefronts per SIMD.
// Measured against the head-128 kernel on padded rows: 16 x 16 heads of 577, size 64, fp16: 60 -> 33 us (660 TFLOP/s); 16 heads
// of 4,096: 102 -> 78 (880); 8 heads of 2,048: 43 -> 19; 8 of 128: 8.6 -> 5.2; 4 x 32 of 2,048, causal: 122 -> 79; size 96,
// 8 x 12 heads of 700: 42 -> 34; against the plain masked kernel: 4 x 12 heads of 1,100 with a bias: 135 -> 39, size 128,
// 2 x 12 of 1,001 with a bias: 263 -> 33; 4 x 32 heads of 1,000, padded: 454 -> 79.
#include <algorithm>

#include "device_common.hpp"
#include "kernels.hpp"

namespace hipattn {

namespace narrow {

constexpr int kWaves = 4;

typedef __attribute__((address_space(3))) uint8_t lds_byte;
typedef __attribute__((address_space(3))) uint4_t lds_uint4;
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef short short8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) short4_t lds_short4;
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

template <bool kBf16>
struct Mfma {
    using vec8 = half8_t;
    static __device__ __forceinline__ float16_t mma(vec8 a, vec8 b, float16_t c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ uint32_t cvt2(float lo, float hi) {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2_t){lo, hi}, half2_t));
    }
    static __device__ __forceinline__ float to_float(uint32_t bits) { return f16_bits_to_float((uint16_t)bits); }
    // x + the two halves of w
    static __device__ __forceinline__ float add2(uint32_t w, float x) {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, w), (half2_t){(half_t)1.0f, (half_t)1.0f}, x, false);
    }
    static constexpr float kSafeSum = 32768.0f;  // sixteen probabilities below it all fit fp16
};
template <>
struct Mfma<true> {
    using vec8 = bf16x8_t;
    static __device__ __forceinline__ float16_t mma(vec8 a, vec8 b, float16_t c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ uint32_t cvt2(float lo, float hi) {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2_t){lo, hi}, bf16x2_t));
    }
    static __device__ __forceinline__ float to_float(uint32_t bits) { return bf16_bits_to_float((uint16_t)bits); }
    static __device__ __forceinline__ float add2(uint32_t w, float x) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w), (bf16x2_t){(__bf16)1.0f, (__bf16)1.0f}, x, false);
    }
    static constexpr float kSafeSum = 16777216.0f;
};

// 16 bytes per lane from lane_offset past a wave-uniform address to LDS byte lds_base + 16 * lane (in assembly, because the
// compiler would wait for every load at every use of LDS; the loop waits for them before its barrier)
__device__ __forceinline__ void load_to_lds_16(const uint8_t* base, uint32_t lane_offset, lds_byte* lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(lane_offset), "s"(base), "s"((uint32_t)(uintptr_t)lds_base)
                 : "memory", "m0");
}
__device__ __forceinline__ void wait_and_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Where the 16-byte chunk c of row r of a tile lies in its row in LDS: sixteen lanes that read one chunk of sixteen rows (K)
// and the four rows a transposing read touches (V) meet different banks.  Rows of 128 bytes: two to the width of the
// banks; rows of 192 start in another quarter each, so that only K's need moving.
template <int kDP>
__device__ __forceinline__ int k_place(int r, int c) { return kDP == 64 ? c ^ ((r >> 1) & 7) : kDP == 96 ? c ^ ((r >> 2) & 3) : c ^ (r & 15); }
template <int kDP>
__device__ __forceinline__ int v_place(int r, int c) { return kDP == 64 ? c ^ (((r >> 1) & 1) << 2) : kDP == 96 ? c : c ^ ((r & 3) << 2); }

enum MaskForm {
    kNoMask,
    kBoolean,   // bytes, keys side by side
    kAdditive   // of the operands' type, keys side by side
};

// kDP: head size the kernel is built for; kPad: the call's is smaller (K's missing columns are zeros in LDS, V's whatever
// is there: they give output columns that nobody stores).  kSplit: wavefronts that share 32 query rows, each with every
// kSplit-th 32 keys; their results meet in LDS at the end.
template <bool kBf16, int kDP, int kForm, bool kPad, int kSplit>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(kDP == 64 && kForm == kNoMask ? 3 : 2))) void sdpa_narrow_kernel(SdpaParams p, int q_tiles, int items) {
    constexpr int kTileK = kSplit == 4 ? 128 : 64, kTileQ = 32 * kWaves / kSplit, kParts = kTileK / 32;
    using M = Mfma<kBf16>;
    using vec8 = typename M::vec8;
    constexpr int kChunks = kDP / 8, kRow = kDP * 2, kStage = kTileK * kRow, kSteps = kDP / 16, kOut = kDP / 32;
    constexpr int kLoads = kStage / 1024 / kWaves;  // load instructions per wavefront and tile
    __shared__ __attribute__((aligned(1024))) uint8_t lds[5 * kStage];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, n32 = lane & 31, hi = lane >> 5;
    // workgroup ids go round the eight XCDs: consecutive items (the query tiles of a head, then those of the next head on
    // the same K and V) stay on one and share its L2.  Causal: the longest tiles of eight heads first, so that short ones
    // fill the end (4 x 32 heads of 2,048, size 64: 96 -> 79 us; 4 x 16 of 1,500, size 96: 51 -> 37)
    const int G = p.num_heads_q / p.num_heads_kv, heads = p.batch * p.num_heads_q;
    const int per_xcd = (items + 7) / 8;
    const int item = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (item >= items) return;
    int head = item / q_tiles, q0 = (q_tiles - 1 - item % q_tiles) * kTileQ;
    if (p.causal && heads % 8 == 0) {
        const int mine = heads / 8, at = (int)(blockIdx.x >> 3), group = at / (8 * q_tiles), in_group = at % (8 * q_tiles);
        const int together = min(8, mine - 8 * group);
        head = (int)(blockIdx.x & 7) * mine + 8 * group + in_group % together;
        q0 = (q_tiles - 1 - in_group / together) * kTileQ;
    }
    const int part = wave % kSplit;  // which 32 keys of a tile, where several wavefronts share the rows
    const int g = head % G, b = head / G % p.batch, hkv = head / G / p.batch, h = hkv * G + g;
    const int D = kPad ? p.head_dim : kDP, row_bytes = 2 * D;
    const int64_t q_off = (((int64_t)b * p.num_heads_q + h) * p.len_q) * D;
    const int64_t kv_off = (((int64_t)b * p.num_heads_kv + hkv) * p.len_kv) * row_bytes;
    const uint8_t* const k = (const uint8_t*)p.k + kv_off;
    const uint8_t* const v = (const uint8_t*)p.v + kv_off;
    const int row0 = q0 + 32 * (wave / kSplit), my_row = row0 + n32;
    int tile0 = 0, key_end = p.causal ? min(p.len_kv, q0 + kTileQ) : p.len_kv;
    if constexpr (kForm == kBoolean) {
        if (p.mask_stride[2] == 0) {  // one row of keys for all queries (padding): from the first key attended to the last
            const uint8_t* const keys = (const uint8_t*)p.mask + (int64_t)b * p.mask_stride[0] + (int64_t)h * p.mask_stride[1];
            int first = key_end, last = -1;
            for (int at = 4 * lane; at < p.len_kv; at += 256)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (keys[min(at + e, p.len_kv - 1)] != 0) first = min(first, at + e), last = max(last, min(at + e, p.len_kv - 1));
#pragma unroll
            for (int x = 32; x > 0; x >>= 1) first = min(first, __shfl_xor(first, x, 64)), last = max(last, __shfl_xor(last, x, 64));
            tile0 = __builtin_amdgcn_readfirstlane(min(first, last + 1) / kTileK);
            key_end = __builtin_amdgcn_readfirstlane(last + 1);
        }
    }
    const int tiles = (key_end + kTileK - 1) / kTileK;
    // steps of 32 keys before which this wavefront is done (one without rows only helps to load)
    const int steps = row0 >= p.len_q ? 0 : ((p.causal ? min(key_end, row0 + 32) : key_end) + 31) / 32;

    lds_byte* const k_lds = (lds_byte*)lds;
    lds_byte* const v_lds = k_lds + 3 * kStage;
    if constexpr (kPad) {  // the columns that no load writes
        for (int i = threadIdx.x; i < 3 * kStage / 16; i += 64 * kWaves) ((lds_uint4*)k_lds)[i] = (uint4_t){0u, 0u, 0u, 0u};
        __syncthreads();
    }
    // this lane's part of load instruction i (of kLoads) of a tile: a row of the tile and a chunk of it
    int load_row[kLoads], k_chunk[kLoads], v_chunk[kLoads];
    uint32_t k_off[kLoads], v_off[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
        const int place = 64 * (wave + kWaves * i) + lane;
        load_row[i] = place / kChunks;
        k_chunk[i] = k_place<kDP>(load_row[i], place % kChunks);
        v_chunk[i] = v_place<kDP>(load_row[i], place % kChunks);
        k_off[i] = (uint32_t)(load_row[i] * row_bytes + 16 * k_chunk[i]);
        v_off[i] = (uint32_t)(load_row[i] * row_bytes + 16 * v_chunk[i]);
    }
    auto load_tile = [&](const uint8_t* base, const uint32_t (&off)[kLoads], const int (&chunk)[kLoads], int keys, lds_byte* stage)
                         __attribute__((always_inline)) {
        if (keys >= kTileK) {
#pragma unroll
            for (int i = 0; i < kLoads; i++)
                if (!kPad || 8 * chunk[i] < D) load_to_lds_16(base, off[i], stage + (wave + kWaves * i) * 1024);
        } else {  // (rows past the end repeat the last key: they are masked)
#pragma unroll
            for (int i = 0; i < kLoads; i++)
                if (!kPad || 8 * chunk[i] < D)
                    load_to_lds_16(base, off[i] - (uint32_t)(max((kPad ? load_row[i] : (int)off[i] / kRow) - (keys - 1), 0) * row_bytes), stage + (wave + kWaves * i) * 1024);
        }
    };
    const int tile_bytes = kTileK * row_bytes;
    const uint8_t* k_src = k + (int64_t)tile0 * tile_bytes;  // the next tile of K and of V to load
    const uint8_t* v_src = v + (int64_t)tile0 * tile_bytes;
    int k_keys = p.len_kv - tile0 * kTileK, v_keys = k_keys;
    auto load_k = [&](lds_byte* stage) __attribute__((always_inline)) {
        load_tile(k_src, k_off, k_chunk, k_keys, stage);
        k_src += tile_bytes, k_keys -= kTileK;
    };
    auto load_v = [&](lds_byte* stage) __attribute__((always_inline)) {
        load_tile(v_src, v_off, v_chunk, v_keys, stage);
        v_src += tile_bytes, v_keys -= kTileK;
    };
    if (tile0 < tiles) {
        load_k(k_lds);
        load_v(v_lds);
        if (tile0 + 1 < tiles) load_k(k_lds + kStage);
    }

    vec8 qf[kSteps];  // Q^T: lane (n32, hi) holds row n32, columns 16 i + 8 hi .. + 7, times scale * log2(e)
    {
        const float c = p.scale * kLog2e;
        const uint16_t* const row = (const uint16_t*)p.q + q_off + (int64_t)min(my_row, p.len_q - 1) * D + 8 * hi;
#pragma unroll
        for (int i = 0; i < kSteps; i++) {
            uint4_t raw = {0u, 0u, 0u, 0u};
            if (!kPad || 16 * i + 8 * hi < D) raw = *(const uint4_t*)(row + 16 * i);
            uint4_t x;
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = M::cvt2(M::to_float(raw[e] & 0xffffu) * c, M::to_float(raw[e] >> 16) * c);
            qf[i] = __builtin_bit_cast(vec8, x);
        }
    }
    // K fragment of key half and k-step i: chunk 2 i + hi of row n32; V^T fragment of 16 keys ks and output tile dt: two
    // transposing reads of four rows each, eight rows apart (lane i of a group of sixteen addresses row i / 4, columns
    // 4 (i % 4) .. + 3 and receives column i of the four rows)
    // (chunk 2 i + hi moves by an exclusive or, so that every k-step's place is the first one's ^ 32 i in rows of 128 and 256 bytes, and
    // within 64 bytes in those of 192)
    const int k_at0 = n32 * kRow + 16 * k_place<kDP>(n32, hi);
    auto k_at = [&](int i) __attribute__((always_inline)) -> int { return kDP != 96 ? k_at0 ^ (32 * i) : (k_at0 ^ (32 * (i & 1))) + 64 * (i >> 1); };
    int v_at[kOut];
    {
        const int grp = lane >> 4, i16 = lane & 15, row = 4 * (grp >> 1) + (i16 >> 2);
#pragma unroll
        for (int dt = 0; dt < kOut; dt++) v_at[dt] = row * kRow + 16 * v_place<kDP>(row, 4 * dt + 2 * (grp & 1) + ((i16 & 3) >> 1)) + 8 * (i16 & 1);
    }
    // The reference of a row's exponents, negated: where the accumulator of its scores starts or, with an additive mask, a
    // part of what the mask adds: fma(mask, log2(e), -reference) is rounded once, so that a constant added to a whole row,
    // which must not change it, costs its scores nothing.  Scores start from that sum or, at size 64, have it added to
    // them (16 heads of 4,096: 138 us against 153; size 96, 2 x 16 of 2,048: 84.5 against 82.9; size 128: 40.0 against 33.0).
    constexpr bool kMaskStarts = kForm == kAdditive && kDP != 64;
    float16_t neg_ref;  // (zero with an additive mask)
    float neg_ref_add = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) neg_ref[r] = 0.f;
    float16_t o[kOut];
#pragma unroll
    for (int dt = 0; dt < kOut; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[dt][r] = 0.f;
    float l_run = 0.f;       // this lane's half of the row's sum
    bool started = false;    // the row has met a key that it attends

    // exponents of the softmax of 32 keys, from `start` on: register r is key 8 (r / 4) + 4 hi + r % 4 of the half
    auto scores = [&](const lds_byte* stage, int half, float16_t& s, const float16_t& start) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kSteps; i++)
            s = M::mma(__builtin_bit_cast(vec8, *(const lds_uint4*)(stage + k_at(i) + half * 32 * kRow)), qf[i], i == 0 ? start : s);
    };
    // the mask of a step for this lane's row, of step t or, where scores start from it, of the one after it: words of four
    // keys (8 g + 4 hi .. + 3)
    constexpr int kMaskWords = kForm == kAdditive ? 8 : kForm == kBoolean ? 4 : 1;
    uint32_t mask[kMaskWords];
    const uint8_t* mask_row = nullptr;
    if constexpr (kForm != kNoMask) {
        constexpr int esz = kForm == kBoolean ? 1 : 2;
        mask_row = (const uint8_t*)p.mask + ((int64_t)b * p.mask_stride[0] + (int64_t)h * p.mask_stride[1] +
                                             (int64_t)min(my_row, p.len_q - 1) * p.mask_stride[2]) * esz;
    }
    auto load_mask = [&](int t) __attribute__((always_inline)) {
        if constexpr (kForm != kNoMask) {
            constexpr int esz = kForm == kBoolean ? 1 : 2;
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) {
                const int key = 32 * t + 8 * g4 + 4 * hi;
                uint32_t w[esz] = {};
                if (key + 4 <= p.len_kv) {
                    __builtin_memcpy(w, mask_row + (int64_t)key * esz, 4 * esz);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)  // (keys past the end: masked anyway)
                        if (key + e < p.len_kv) {
                            if constexpr (esz == 1)
                                w[0] |= (uint32_t)mask_row[key + e] << (8 * e);
                            else
                                w[e >> 1] |= (uint32_t)((const uint16_t*)mask_row)[key + e] << (16 * (e & 1));
                        }
                }
#pragma unroll
                for (int x = 0; x < esz; x++) mask[esz * g4 + x] = w[x];
            }
        }
    };
    auto addend = [&](int r) __attribute__((always_inline)) -> float {
        return fmaf(M::to_float((mask[r >> 1] >> (16 * (r & 1))) & 0xffffu), kLog2e, neg_ref_add);
    };
    auto start_scores = [&](float16_t& s) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = addend(r);
    };
    constexpr int kNext = kSplit == 1 ? 1 : kParts;  // from one step of a wavefront to its next
    bool stale = false;  // (kMaskStarts) the reference has moved far from where the next step's scores were started
    vec8 pf[2], vf[2][kOut];  // probabilities of the step before and the V^T fragments that they meet
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
        pf[ks] = __builtin_bit_cast(vec8, (uint4_t){0u, 0u, 0u, 0u});
#pragma unroll
        for (int dt = 0; dt < kOut; dt++) vf[ks][dt] = pf[ks];
    }
    auto accumulate = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < 2; ks++)
#pragma unroll
            for (int dt = 0; dt < kOut; dt++) o[dt] = M::mma(vf[ks][dt], pf[ks], o[dt]);
    };
    // One step: its exponentials, and beside them on the matrix core O^T += V^T P^T of the step before and the scores of the next.
    auto step = [&](int t, float16_t& s, float16_t& s_next, const lds_byte* k_this, const lds_byte* k_next, int half_next, const lds_byte* v_stage, int half)
                    __attribute__((always_inline)) {
        if constexpr (kForm == kBoolean) {
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = ((mask[r >> 2] >> (8 * (r & 3))) & 0xffu) != 0 ? s[r] : -INFINITY;
        }
        if constexpr (kForm == kAdditive && !kMaskStarts) {
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] += addend(r);
        }
        if constexpr (kForm != kNoMask && !kMaskStarts) {
            if (t + kNext < steps) load_mask(t + kNext);
        }
        auto scores_again = [&]() __attribute__((always_inline)) {
            load_mask(t);
            float16_t start;
            start_scores(start);
            scores(k_this, half, s, start);
        };
        if constexpr (kMaskStarts) {
            if (stale) {
                scores_again();
                if (t + kNext < steps) load_mask(t + kNext);
                stale = false;
            }
        }
        auto cut_edges = [&]() __attribute__((always_inline)) {
            if (32 * t + 32 > p.len_kv || (p.causal && 32 * t + 31 > row0)) {
                const int end = (p.causal ? min(p.len_kv, my_row + 1) : p.len_kv) - 32 * t - 4 * hi;
#pragma unroll
                for (int r = 0; r < 16; r++) s[r] = 8 * (r >> 2) + (r & 3) < end ? s[r] : -INFINITY;
            }
        };
        cut_edges();
        constexpr bool kStartEarly = kDP < 128;  // (size 128 has no registers for it until half of the step is done)
        auto start_next = [&]() __attribute__((always_inline)) {  // (after the last step: unused)
            start_scores(s_next);
            if (t + 2 * kNext < steps) load_mask(t + 2 * kNext);
        };
        if constexpr (kMaskStarts && kStartEarly) start_next();
        vec8 pn[2];
        auto probabilities = [&](int ks) __attribute__((always_inline)) -> float {  // of sixteen keys; returns their sum
            float sum = 0.f;
            uint4_t w;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                w[e] = M::cvt2(fast_exp2(s[8 * ks + 2 * e]), fast_exp2(s[8 * ks + 2 * e + 1]));
                sum = M::add2(w[e], sum);
            }
            pn[ks] = __builtin_bit_cast(vec8, w);
            return sum;
        };
        // In this order (the compiler would read each fragment right before its use and wait for it every time), with the
        // matrix instructions spread over the vector ones
        vec8 kf[kSteps];
#pragma unroll
        for (int i = 0; i < kSteps; i++) kf[i] = __builtin_bit_cast(vec8, *(const lds_uint4*)(k_next + k_at(i) + half_next * 32 * kRow));
        __builtin_amdgcn_sched_barrier(0);
        accumulate();
        float sum = probabilities(0);
#pragma unroll
        for (int x = 0; x < 2 * kOut; x++) {
            __builtin_amdgcn_sched_group_barrier(0x2, 24 / (2 * kOut), 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kMaskStarts && !kStartEarly) start_next();
#pragma unroll
        for (int ks = 0; ks < 2; ks++)
#pragma unroll
            for (int dt = 0; dt < kOut; dt++) {
                const lds_byte* const at = v_stage + v_at[dt] + (2 * half + ks) * 16 * kRow;
                const short4_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)at);
                const short4_t a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(at + 8 * kRow));
                const short8_t a = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
                vf[ks][dt] = __builtin_bit_cast(vec8, a);
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kSteps; i++) s_next = M::mma(kf[i], qf[i], i == 0 && !kMaskStarts ? neg_ref : s_next);  // (after the last step: unused)
        sum += probabilities(1);
#pragma unroll
        for (int x = 0; x < kSteps; x++) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, 24 / kSteps, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        // The reference stays while every sum says that no probability can have overflowed; otherwise, and for the first
        // keys of a row, it moves to the largest score (all in units of exponents to base 2).
        if (__builtin_amdgcn_ballot_w64(!started || !(sum < M::kSafeSum)) != 0) {
            // An additive mask says "not this key" by a large negative number as well as by -inf, and a reference taken from such keys
            // leaves the scores of the others, 94,500 above it with fp16's lowest value, rounded to 2^-7.  So after a move by
            // more than 2^9, which leaves nothing of what a row has summed up, its scores are computed again (to 2^-15) and its
            // reference is chosen again, off by the rounding of the last one: 2^-24 of it, so that 10^38 takes six moves.
            constexpr float kFar = 512.0f;
            auto move = [&]() __attribute__((always_inline)) -> bool {
                float top = -INFINITY;
#pragma unroll
                for (int r = 0; r < 16; r++) top = fmaxf(top, s[r]);
                const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(top), __float_as_uint(top), false, false);
                top = fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1]));
                const bool seen = top != -INFINITY;
                if (__builtin_amdgcn_ballot_w64(top > 8.0f || (seen && !started)) == 0) return false;
                float delta = started ? fmaxf(top, 0.f) : (seen ? top : 0.f);
                if constexpr (kForm == kAdditive) {  // by what the new reference is, rounded, as the next steps will see it
                    const float moved = neg_ref_add - delta;
                    delta = neg_ref_add - moved;
                    neg_ref_add = moved;
                }
                const float alpha = fast_exp2(-fmaxf(delta, 0.f));
                l_run *= alpha;
#pragma unroll
                for (int dt = 0; dt < kOut; dt++) o[dt] *= alpha;
                s -= delta;
                started = started || seen;
                if constexpr (kForm != kAdditive || kMaskStarts) s_next -= delta;
                if constexpr (kForm == kAdditive) {
                    const bool far = fabsf(delta) > kFar;
                    started = started && !far;
                    return __builtin_amdgcn_ballot_w64(far) != 0;
                } else {
                    neg_ref -= delta;
                    return false;
                }
            };
            bool again = move();
            if constexpr (kForm == kAdditive) {
                const bool far = again;
                for (int tries = 0; again && tries < 8; tries++) {
                    scores_again();
                    cut_edges();
                    again = move();
                }
                constexpr int kLoaded = kMaskStarts ? 2 * kNext : kNext;  // which step's mask has been overwritten
                if (far && t + kLoaded < steps) load_mask(t + kLoaded);
                if constexpr (kMaskStarts) stale = far;
            }
            sum = probabilities(0) + probabilities(1);
        }
        l_run += sum;
        pf[0] = pn[0], pf[1] = pn[1];
    };

    float16_t s0, s1;
    lds_byte *k_now, *k_next, *k_fill, *v_now, *v_fill;
    const int t0 = kParts * tile0 + part;
    // One tile: K of the next tile and V of this one, loaded an iteration ago, are there for every wavefront, and the
    // stages that are filled now were last read before the barrier
    auto iteration = [&](int j, float16_t& a, float16_t& b) __attribute__((always_inline)) {
        if (j > tile0) wait_and_barrier();
        if (j + 2 < tiles) load_k(k_fill);
        if (j + 1 < tiles) load_v(v_fill);
        const int t = kParts * j + part;
        if constexpr (kSplit == 1) {
            if (t < steps) step(t, a, b, k_now, k_now, 1, v_now, 0);
            if (t + 1 < steps) step(t + 1, b, a, k_now, k_next, 0, v_now, 1);
        } else {
            if (t < steps) step(t, a, b, k_now, k_next, part, v_now, part);
        }
        lds_byte *const k_done = k_now, *const v_done = v_now;
        k_now = k_next, k_next = k_fill, k_fill = k_done;
        v_now = v_fill, v_fill = v_done;
    };
    k_now = k_lds, k_next = k_lds + kStage, k_fill = k_lds + 2 * kStage, v_now = v_lds, v_fill = v_lds + kStage;
    if (t0 < steps) load_mask(t0);
    if constexpr (kMaskStarts) {
        start_scores(s0);
        if (t0 + kNext < steps) load_mask(t0 + kNext);
    }
    wait_and_barrier();
    scores(k_now, part, s0, kMaskStarts ? s0 : neg_ref);
    if constexpr (kSplit == 1) {
        for (int j = tile0; j < tiles; j++) iteration(j, s0, s1);
    } else {
        for (int j = tile0; j < tiles; j += 2) {
            iteration(j, s0, s1);
            if (j + 1 < tiles) iteration(j + 1, s1, s0);
        }
    }
    accumulate();

    const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
    float l = __uint_as_float(both[0]) + __uint_as_float(both[1]);
    uint16_t* const out = (uint16_t*)p.out + q_off + (int64_t)my_row * D;
    // x[0 .. 7]: columns 32 dt + 8 gg + 4 hi + r % 4 (r < 4) and eight further; lanes l and l + 32 exchange halves so that
    // each stores eight in a row
    auto store = [&](const float (&x)[8], int dt, int gg) __attribute__((always_inline)) {
        const auto a = __builtin_amdgcn_permlane32_swap(M::cvt2(x[0], x[1]), M::cvt2(x[4], x[5]), false, false);
        const auto c = __builtin_amdgcn_permlane32_swap(M::cvt2(x[2], x[3]), M::cvt2(x[6], x[7]), false, false);
        const int d = 32 * dt + 8 * (gg + hi);
        if (my_row < p.len_q && (!kPad || d < D)) *(uint4_t*)(out + d) = (uint4_t){a[0], c[0], a[1], c[1]};
    };
    if constexpr (kSplit == 1) {
        const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
        for (int dt = 0; dt < kOut; dt++)
#pragma unroll
            for (int gg = 0; gg < 4; gg += 2) {
                float x[8];
#pragma unroll
                for (int r = 0; r < 8; r++) x[r] = o[dt][4 * gg + r] * inv;
                store(x, dt, gg);
            }
    } else {
        typedef __attribute__((address_space(3))) float lds_float;
        lds_float* const shares = (lds_float*)lds;  // [wavefront][reference, sum, accumulators][lane]
        constexpr int kShare = (16 * kOut + 2) * 64;
        static_assert(kWaves * kShare * 4 <= 5 * kStage, "the shares take the place of the stages");
        __syncthreads();  // (every wavefront is done with the stages, and no load is under way)
        lds_float* const mine = shares + wave * kShare + lane;
        mine[0] = started ? -(kForm == kAdditive ? neg_ref_add : neg_ref[0]) : -INFINITY;
        mine[64] = l;
#pragma unroll
        for (int dt = 0; dt < kOut; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) mine[(2 + 16 * dt + r) * 64] = o[dt][r];
        __syncthreads();
        const lds_float* const first = shares + (wave - part) * kShare + lane;
        float f[kSplit], top = -INFINITY, total = 0.f;
#pragma unroll
        for (int x = 0; x < kSplit; x++) f[x] = first[x * kShare], top = fmaxf(top, f[x]);
#pragma unroll
        for (int x = 0; x < kSplit; x++) {
            f[x] = f[x] == -INFINITY ? 0.f : fast_exp2(f[x] - top);
            total = fmaf(f[x], first[x * kShare + 64], total);
        }
        const float inv = total > 0.f ? 1.0f / total : 0.f;
#pragma unroll
        for (int i = 0; i < 2 * kOut; i++) {  // eight accumulators each: the sharers take turns
            if (i % kSplit != part) continue;
            float x[8];
#pragma unroll
            for (int r = 0; r < 8; r++) {
                float sum = 0.f;
#pragma unroll
                for (int w = 0; w < kSplit; w++) sum = fmaf(f[w], first[w * kShare + (2 + 8 * i + r) * 64], sum);
                x[r] = sum * inv;
            }
            store(x, i / 2, 2 * (i % 2));
        }
    }
}

// Wavefronts that share 32 query rows, from the time the busiest compute unit would take, in microseconds: per step 0.30 and a
// share for every workgroup beside each other on it (fitted: size 64 0.41 / 0.59 / 0.74 with one to three, size 128 0.64 / 0.96
// with one and two), a fifth more where every step has a barrier, and what a workgroup costs however few its steps are.
// Measured around the lines it draws, with 1 / 2 / 4: 8 heads of 2,048, size 64: 29.5 / 20.1 / 19.8 us; 12 of 800: 14.2 / 10.8 /
// 12.0; 48 of 800: 18.4 / 16.7 / 26.6; 96 of 800: 24.8 / 27.7 / 49.2; 96 of 130: 6.4 / 7.3 / 7.7; 64 of 77 rows and 1,024 keys:
// 16.2 / 12.0 / 10.1; 16 of 4,096: 80 / 88 / 121; size 128, 12 of 1,000: 25.2 / 17.2 / 27.7; 12 of 500, causal: 14.6 / 11.2 / 10.2;
// 16 x 32 of 150, causal, three rounds of workgroups where two share the rows: 18.5 / 24.2 (23.2 in the head-128 kernel).
struct Split {
    int split;
    double cost;
};
Split choose_split(const SdpaParams& p) {
    Split best{1, 0};
    for (int split = 1; split <= 4; split *= 2) {
        const int64_t groups = (int64_t)p.batch * p.num_heads_q * ((p.len_q + 128 / split - 1) / (128 / split));
        const int64_t per_cu = (groups + 255) / 256;
        const int resident = p.head_dim <= 64 ? (split == 4 || p.mask ? 2 : 3) : (split == 4 ? 1 : 2);
        const int steps = ((p.len_kv + 31) / 32 + split - 1) / split;  // (causal: of the longest)
        const double share = p.head_dim <= 64 ? 0.14 : p.head_dim <= 96 ? 0.21 : 0.32;
        const auto round = [&](int n) {
            const double fixed = split == 1 ? (p.head_dim <= 64 ? 1.5 : 2.5 * n - 1.0) : split == 2 ? 2.2 : 2.5 + 0.9 * n;
            return steps * (0.30 + share * n) * (split == 1 ? 1.0 : 1.2) + fixed;
        };
        double cost = (double)(per_cu / resident) * round(resident) + (per_cu % resident ? round((int)(per_cu % resident)) : 0);
        if (split == 2 && p.head_dim > 96) cost += 2.2 * (double)((per_cu - 1) / resident);
        if (best.cost == 0 || cost < best.cost) best = {split, cost};
    }
    return best;
}

template <bool kBf16, int kDP, int kForm, int kSplit>
void launch(const SdpaParams& p, hipStream_t stream) {
    constexpr int kRows = 32 * kWaves / kSplit;
    const int q_tiles = (p.len_q + kRows - 1) / kRows, items = p.batch * p.num_heads_q * q_tiles;
    const dim3 grid((unsigned)((items + 7) / 8 * 8)), block(64 * kWaves);
    if constexpr (kDP != 64)
        if (p.head_dim < kDP) {
            hipLaunchKernelGGL((sdpa_narrow_kernel<kBf16, kDP, kForm, true, kSplit>), grid, block, 0, stream, p, q_tiles, items);
            return;
        }
    hipLaunchKernelGGL((sdpa_narrow_kernel<kBf16, kDP, kForm, false, kSplit>), grid, block, 0, stream, p, q_tiles, items);
}

template <bool kBf16, int kDP, int kForm>
void launch(const SdpaParams& p, hipStream_t stream) {
    const int wanted = sdpa_narrow_split_option(), split = wanted > 0 ? wanted : choose_split(p).split;
    if (split == 1)
        launch<kBf16, kDP, kForm, 1>(p, stream);
    else if (split < 4)
        launch<kBf16, kDP, kForm, 2>(p, stream);
    else
        launch<kBf16, kDP, kForm, 4>(p, stream);
}

template <bool kBf16, int kDP>
void launch(const SdpaParams& p, hipStream_t stream) {
    if (!p.mask)
        launch<kBf16, kDP, kNoMask>(p, stream);
    else if (p.mask_dtype == HIPATTN_U8)
        launch<kBf16, kDP, kBoolean>(p, stream);
    else
        launch<kBf16, kDP, kAdditive>(p, stream);
}

}  // namespace narrow

// 16-bit operands at 16-byte aligned addresses; no mask, or one whose keys lie side by side, boolean or of the operands' type.
static bool sdpa_narrow_supported(const SdpaParams& p) {
    if (p.dtype != HIPATTN_F16 && p.dtype != HIPATTN_BF16) return false;
    if (p.head_dim != 64 && (p.head_dim < 72 || p.head_dim > 128 || p.head_dim % 8 != 0)) return false;
    if (p.mask && (p.mask_stride[3] != 1 || (p.mask_dtype != HIPATTN_U8 && p.mask_dtype != p.dtype))) return false;
    const int64_t tiles = (int64_t)p.batch * p.num_heads_q * (((int64_t)p.len_q + 31) / 32);
    return p.len_q > 0 && p.len_kv > 0 && p.batch > 0 && tiles < (1 << 30) &&
           (((uintptr_t)p.q | (uintptr_t)p.k | (uintptr_t)p.v | (uintptr_t)p.out) & 15) == 0;
}

// Head sizes above 64 share with the kernel of flash_prefill.hip, whose workgroup has a compute unit to itself, takes 256 rows
// and needs some 1.25 us for 64 keys, 1.5 to 1.8 with the chip full, and 4 to 7 besides.  Above 96 it is faster where it fills the chip (4 x 32
// heads of 2,048, causal: 136 against 142 us; 4 x 8 of 1,300: 35 against 42) and slower on small calls (8 heads of 2,048: 42 against 28;
// 12 of 500, causal: 18.4 against 10.2; 8 of 48: 7.4 against 5.6) and with a mask.  Up to 96 it computes 128 columns all the
// same and is the faster one only without a mask or the causal flag, where its workgroups come out as one round and these as a
// little more than one (size 80, 2 x 12 heads of 1,390: 33.2 against 35.2; 2 x 16 of 1,500: 38.0 and 38.3; 4 x 16 of 1,024: 33.8 against
// 31.7; 8 x 12 of 700: 42 against 33).
static bool sdpa_narrow_preferred(const SdpaParams& p) {
    if (p.head_dim == 64 || (p.head_dim <= 96 && (p.mask || p.causal))) return true;
    // (additive masks: 4 x 8 heads of 1,024 33 against 50 us; 4 x 32 of 2,048, four rounds of workgroups: 368 against 375)
    if (p.mask) return p.mask_dtype == HIPATTN_U8 || (int64_t)p.batch * p.num_heads_q * ((p.len_q + 127) / 128) <= 512;
    const int G = p.num_heads_q / p.num_heads_kv, q_tiles = (p.len_q + 127) / 128;
    const int64_t groups = (int64_t)p.batch * p.num_heads_kv * (G % 2 == 0 ? G / 2 * q_tiles : G * ((q_tiles + 1) / 2));
    const int64_t rounds = (groups + 255) / 256;
    const double tiles = (p.len_kv + 63) / 64, cost = narrow::choose_split(p).cost;
    if (p.head_dim <= 96) return cost < 1.02 * (double)rounds * (tiles * (1.25 + 0.55 / 128 * (double)std::clamp<int64_t>(groups - 128, 0, 128)) + 5.0);
    return cost < 0.9 * (double)rounds * (tiles * (groups > 128 ? 1.5 : 1.25) + (rounds > 1 ? 7.0 : 4.0));
}

// (sdpa_padded_rows = 0 leaves head sizes below 128 to the plain kernels)
bool sdpa_takes_narrow(const SdpaParams& p, bool flash) {
    const int option = sdpa_narrow_option();
    if (option == 0 || !sdpa_narrow_supported(p)) return false;
    return option == 2 || (flash ? sdpa_narrow_preferred(p) : sdpa_padded_rows_enabled());
}

hipError_t launch_sdpa_narrow(const SdpaParams& p, hipStream_t stream, const KernelProbe& probe) {
    if (probe.before) (void)hipEventRecord(probe.before, stream);
    if (p.dtype == HIPATTN_BF16)
        p.head_dim == 64 ? narrow::launch<true, 64>(p, stream) : p.head_dim <= 96 ? narrow::launch<true, 96>(p, stream) : narrow::launch<true, 128>(p, stream);
    else
        p.head_dim == 64 ? narrow::launch<false, 64>(p, stream) : p.head_dim <= 96 ? narrow::launch<false, 96>(p, stream) : narrow::launch<false, 128>(p, stream);
    const hipError_t e = hipGetLastError();
    if (probe.after) (void)hipEventRecord(probe.after, stream);
    return e;
}

}  // namespace hipattn
