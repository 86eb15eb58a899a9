// Dense attention with fp32 operands on the fp32 matrix cores: v_mfma_f32_16x16x4_f32, which multiplies and
// accumulates in fp32 throughout.
//
// A wavefront owns 16 * kNT query rows of one head and a share of the keys; the wavefronts of a workgroup
// take the same rows and different keys and add up their results at the end.  Nothing is shared in the loop:
// no LDS, no barrier.  K and V fragments come straight from global memory (an XCD's L2 holds the heads it
// works on) in 16-byte pieces:
//   S^T = K Q^T   A = K: lane (key n, quarter q) loads K[key][16 i + 4 q ..+3], four MFMAs of the contraction
//                 columns {4 q + t}; Q^T is held in registers with the same permutation
//   O^T = V^T P^T the accumulator of S^T (lane (row n, q), register r: key 4 q + r) is the B operand as it
//                 stands; A = V^T: the lane loads V[key 4 q + r][64 c + 4 n ..+3], so four MFMAs give the output
//                 columns 64 c + 4 m + t
// What bounds it: fp32 MFMAs run on the vector ALU's own multipliers.  A wavefront of v_fma or v_exp beside one of
// these MFMAs on a SIMD takes the sum of the two times (96 + 122 -> 208 us, where bf16 MFMAs overlap: 108 + 119 ->
// 153), so every vector instruction in the loop adds to the 32 cycles of each MFMA and the loop is built to have few:
// addresses advance in scalar registers, and the exponents' reference is the maximum of the first keys attended for
// as long as no exponent passes 2^kSafe above it (fp32 has the range; the sums are the same), so that no maximum is
// taken per step.  Measured: 2 x 8 heads of 2,048 tokens at head size 64: 133 us = 129 TFLOP/s (a large fp32 matrix
// product reaches 149 on this card); 8 x 12 heads of 384, padded: 1,660 us in the shape-generic kernel -> 37; 8 heads of
// 128, causal: 55 -> 5.4.
#include "attend_row.hpp"
#include "kernels.hpp"

namespace hipattn {

namespace {

constexpr float kSafeExp = 0x1p60f;  // a step whose exponentials stay below keeps its reference (their sums stay far from overflow)

// max / sum over the four lanes (n, n + 16, n + 32, n + 48) that share a query row
template <typename F>
__device__ __forceinline__ float across_quarters(float x, F f) {
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
    a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return f(__uint_as_float(a[0]), __uint_as_float(a[1]));
}

// What a call's attention mask is to the kernel: a form each, so that the loop holds one form's few instructions.
enum MaskForm {
    kNoMask,
    kBoolean,   // bytes, keys side by side: four per lane and step in one word
    kFloat,     // fp32, keys side by side
    kAnyMask    // every other type and stride: one load per key
};

// The mask of four consecutive keys of a row, fetched a step ahead: the four bytes (kBoolean) or four addends.
template <int kForm>
__device__ __forceinline__ uint4_t fetch_mask4(const uint8_t* row, int64_t key_stride, int dtype, int key, int len_kv) {
    uint4_t raw = {0u, 0u, 0u, 0u};
    if (kForm != kAnyMask && key + 3 < len_kv) {
        if (kForm == kBoolean)
            __builtin_memcpy(&raw, row + key, 4);
        else
            __builtin_memcpy(&raw, row + 4 * (int64_t)key, 16);
        return raw;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {  // (keys past the end repeat the last one: they are masked anyway)
        const int64_t at = (int64_t)min(key + e, len_kv - 1) * key_stride;
        if (kForm == kBoolean)
            raw[0] |= (uint32_t)row[at] << (8 * e);
        else if (kForm == kFloat)
            raw[e] = ((const uint32_t*)row)[at];
        else
            raw[e] = __float_as_uint(dtype == HIPATTN_U8 ? (row[at] ? 0.f : -INFINITY) : load_scalar(row, at, dtype));
    }
    return raw;
}

// kDP: the head size the kernel is built for (kPad: the call's is smaller, the missing columns of Q and K are
// zeros); kNT: row tiles of 16 per wavefront.  snake: see launch().
// (Three wavefronts to a SIMD at one row tile of size 128, which 168 registers allow: 3 x 12 heads of 300 with a mask 29.4 us, with two 37.3.)
template <int kDP, int kNT, int kForm, bool kPad>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(kDP == 128 && kNT == 1 && !kPad ? 3 : 2))) void sdpa_f32_kernel(SdpaParams p, int q_tiles, int items, int snake) {
    constexpr int kC = kDP / 64, kI = kDP / 16, kStep = 16, kRows = 16 * kNT;
    constexpr bool kAdds = kForm == kFloat || kForm == kAnyMask;  // scores carry scale and mask; else the exponent's multiply-add scales
    extern __shared__ __align__(16) uint8_t lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int lane = threadIdx.x & 63, n = lane & 15, quarter = lane >> 4;
    // workgroup ids go round the eight XCDs: consecutive items (the query tiles of one head, then those of the
    // same head of the next batch entry) stay on one, so that its L2 serves their K and V, and every XCD has
    // heads of all batch entries, whose keys a padding mask may leave of very different length
    const int per_xcd = (items + 7) / 8;
    const int item = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (item >= items) return;
    const int hb = item / q_tiles, at = item % q_tiles;
    const int row0 = (snake && (hb & 1) ? at : q_tiles - 1 - at) * kRows;
    const int b = hb % p.batch, h = hb / p.batch, bh = b * p.num_heads_q + h;
    const int D = kPad ? p.head_dim : kDP;
    const int64_t kv_off = ((int64_t)b * p.num_heads_kv + h / (p.num_heads_q / p.num_heads_kv)) * p.len_kv * D;
    const float* const q = (const float*)p.q + (int64_t)bh * p.len_q * D;
    const float* const k = (const float*)p.k + kv_off;
    const float* const v = (const float*)p.v + kv_off;
    const int key_end = p.causal ? min(p.len_kv, row0 + kRows) : p.len_kv;
    const int steps = (key_end + kStep - 1) / kStep;
    const int first = steps * wave / waves, last = steps * (wave + 1) / waves;
    const float c = p.scale * kLog2e;

    float4_t qf[kNT][kI];
#pragma unroll
    for (int nt = 0; nt < kNT; nt++) {
        const float* const row = q + (int64_t)min(row0 + 16 * nt + n, p.len_q - 1) * D;
#pragma unroll
        for (int i = 0; i < kI; i++) {
            const int d = 16 * i + 4 * quarter;
            qf[nt][i] = kPad && d >= D ? (float4_t){0.f, 0.f, 0.f, 0.f} : *(const float4_t*)(row + d);
        }
    }
    // a step's addresses: a base that advances in scalar registers plus a lane's own offset in bytes, which is set for good
    // here and once more for a last step that ends beyond the keys (its missing rows repeat the last key)
    uint32_t k_at, v_at[4];
    auto lane_offsets = [&](int key0) __attribute__((always_inline)) {
        const int most = p.len_kv - 1 - key0;
        k_at = (uint32_t)(min(n, most) * D + 4 * quarter) * 4u;
#pragma unroll
        for (int r = 0; r < 4; r++) v_at[r] = (uint32_t)(min(4 * quarter + r, most) * D + 4 * n) * 4u;
    };
    float4_t kf[kI], vf[4][kC];
    auto fetch_k = [&](int step) __attribute__((always_inline)) {
        const uint8_t* const base = (const uint8_t*)(k + (int64_t)step * (kStep * D));
#pragma unroll
        for (int i = 0; i < kI; i++) {
            const int d = 16 * i + 4 * quarter;
            kf[i] = kPad && d >= D ? (float4_t){0.f, 0.f, 0.f, 0.f} : *(const float4_t*)(base + k_at + 64 * i);
        }
    };
    auto fetch_v = [&](int step) __attribute__((always_inline)) {
        const uint8_t* const base = (const uint8_t*)(v + (int64_t)step * (kStep * D));
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int cc = 0; cc < kC; cc++)  // (columns past the head size repeat others: output columns nobody stores)
                vf[r][cc] = *(const float4_t*)(base + (v_at[r] + (kPad && 64 * cc + 4 * n >= D ? -16 * n : 256 * cc)));
    };
    uint4_t mask[kNT];
    const uint8_t* mask_row[kNT];
    if constexpr (kForm != kNoMask) {
        const int esz = p.mask_dtype == HIPATTN_U8 ? 1 : dtype_bytes(p.mask_dtype);
#pragma unroll
        for (int nt = 0; nt < kNT; nt++)
            mask_row[nt] = (const uint8_t*)p.mask + ((int64_t)b * p.mask_stride[0] + (int64_t)h * p.mask_stride[1] +
                                                     (int64_t)min(row0 + 16 * nt + n, p.len_q - 1) * p.mask_stride[2]) * esz;
    }
    auto fetch_mask = [&](int step) __attribute__((always_inline)) {
        if constexpr (kForm != kNoMask) {
#pragma unroll
            for (int nt = 0; nt < kNT; nt++)
                mask[nt] = fetch_mask4<kForm>(mask_row[nt], p.mask_stride[3], p.mask_dtype, step * kStep + 4 * quarter, p.len_kv);
        }
    };

    float4_t o[kC][4][kNT];
    float m[kNT], l[kNT];  // the exponents' reference (-inf until a key is attended) and this lane's share of the row sum
#pragma unroll
    for (int nt = 0; nt < kNT; nt++) {
        m[nt] = -INFINITY, l[nt] = 0.f;
#pragma unroll
        for (int cc = 0; cc < kC; cc++)
#pragma unroll
            for (int t = 0; t < 4; t++) o[cc][t][nt] = (float4_t){0.f, 0.f, 0.f, 0.f};
    }
    const bool ragged = steps * kStep > p.len_kv;  // the last step of all ends beyond the keys
    if (first < last) {
        lane_offsets(ragged && first == steps - 1 ? first * kStep : 0);
        fetch_k(first);
        fetch_mask(first);
    }
    for (int step = first; step < last; step++) {
        const int key0 = step * kStep, next = min(step + 1, last - 1);
        uint4_t now[kNT];
        bool attended = true, partly = false;  // a step whose keys are masked for every row is passed over
        if constexpr (kForm != kNoMask) {
            bool any = false, gap = false;
#pragma unroll
            for (int nt = 0; nt < kNT; nt++) {
                now[nt] = mask[nt];
                if constexpr (kForm == kBoolean) {
                    const uint32_t w = now[nt][0];
                    any |= w != 0;
                    gap |= ((w - 0x01010101u) & ~w & 0x80808080u) != 0;  // (one of the four bytes is zero)
                } else {
                    const float4_t x = __builtin_bit_cast(float4_t, now[nt]);
                    // (a NaN masks nothing: it becomes the row's, so not fmaxf, which would pass over it)
                    const auto larger = [](float a, float b) { return __builtin_elementwise_maximum(a, b); };
                    any |= larger(larger(x[0], x[1]), larger(x[2], x[3])) != -INFINITY;
                    gap |= fminf(fminf(x[0], x[1]), fminf(x[2], x[3])) == -INFINITY;
                }
            }
            attended = __builtin_amdgcn_ballot_w64(any) != 0;
            partly = __builtin_amdgcn_ballot_w64(gap) != 0;
            fetch_mask(next);
        }
        // V of this step is on its way while the scores are computed, K of the next one while the exponents and
        // the output are (the fences keep the compiler from sinking the loads to their first use)
        float4_t s[kNT];
        if (attended) {
            fetch_v(step);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int nt = 0; nt < kNT; nt++) s[nt] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < kI; i++)
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int nt = 0; nt < kNT; nt++) s[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i][t], qf[nt][i][t], s[nt], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (ragged && step + 2 == steps) lane_offsets(key0 + kStep);
        fetch_k(next);
        __builtin_amdgcn_sched_barrier(0);
        if (!attended) continue;
        if constexpr (kAdds) {
#pragma unroll
            for (int nt = 0; nt < kNT; nt++)
#pragma unroll
                for (int r = 0; r < 4; r++) s[nt][r] = fmaf(s[nt][r], c, __uint_as_float(now[nt][r]) * kLog2e);
        }
        if (kForm == kBoolean && partly) {
#pragma unroll
            for (int nt = 0; nt < kNT; nt++)
#pragma unroll
                for (int r = 0; r < 4; r++) s[nt][r] = (now[nt][0] >> (8 * r)) & 0xffu ? s[nt][r] : -INFINITY;
        }
        if (kForm != kNoMask && partly) {
            // Value rows of keys that no row of the tile attends (padding: whatever the buffer held) become zeros, so that
            // a zero probability times an infinity or NaN does not send the tile's rows through the slow way below.
#pragma unroll
            for (int r = 0; r < 4; r++) {
                bool has = false;
#pragma unroll
                for (int nt = 0; nt < kNT; nt++) has |= kForm == kBoolean ? ((now[nt][0] >> (8 * r)) & 0xffu) != 0 : __uint_as_float(now[nt][r]) != -INFINITY;
                const bool keep = ((__builtin_amdgcn_ballot_w64(has) >> (16 * quarter)) & 0xffff) != 0;
#pragma unroll
                for (int cc = 0; cc < kC; cc++)
#pragma unroll
                    for (int e = 0; e < 4; e++) vf[r][cc][e] = keep ? vf[r][cc][e] : 0.f;
            }
        }
        if (key0 + kStep > p.len_kv || (p.causal && key0 + kStep - 1 > row0)) {
#pragma unroll
            for (int nt = 0; nt < kNT; nt++) {
                const int end = p.causal ? min(p.len_kv, row0 + 16 * nt + n + 1) : p.len_kv;
#pragma unroll
                for (int r = 0; r < 4; r++) s[nt][r] = key0 + 4 * quarter + r < end ? s[nt][r] : -INFINITY;
            }
        }
        float4_t e[kNT];
        float sum[kNT];
        auto exponentials = [&](int nt) __attribute__((always_inline)) {
            const float ref = m[nt] == -INFINITY ? 0.f : m[nt];
#pragma unroll
            for (int r = 0; r < 4; r++) e[nt][r] = fast_exp2(kAdds ? s[nt][r] - ref : fmaf(s[nt][r], c, -ref));
            sum[nt] = (e[nt][0] + e[nt][1]) + (e[nt][2] + e[nt][3]);
        };
        bool unsafe = false;
#pragma unroll
        for (int nt = 0; nt < kNT; nt++) {
            exponentials(nt);
            unsafe |= !(sum[nt] < kSafeExp) || m[nt] == -INFINITY;
        }
        if (__builtin_amdgcn_ballot_w64(unsafe) != 0) {  // the first keys a row attends, or an exponent out of bounds
#pragma unroll
            for (int nt = 0; nt < kNT; nt++) {
                float top = fmaxf(fmaxf(s[nt][0], s[nt][1]), fmaxf(s[nt][2], s[nt][3]));
                top = across_quarters(top, [](float a, float b) { return fmaxf(a, b); });
                if (!kAdds) top *= c;
                top = fmaxf(top, m[nt]);
                const float alpha = m[nt] == -INFINITY ? 0.f : fast_exp2(m[nt] - top);
                l[nt] *= alpha;
#pragma unroll
                for (int cc = 0; cc < kC; cc++)
#pragma unroll
                    for (int t = 0; t < 4; t++) o[cc][t][nt] *= alpha;
                m[nt] = top;
                exponentials(nt);
            }
        }
#pragma unroll
        for (int nt = 0; nt < kNT; nt++) l[nt] += sum[nt];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int cc = 0; cc < kC; cc++)
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int nt = 0; nt < kNT; nt++)
                        o[cc][t][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[r][cc][t], e[nt][r], o[cc][t][nt], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int nt = 0; nt < kNT; nt++) l[nt] = across_quarters(l[nt], [](float a, float b) { return a + b; });

    if (waves > 1) {  // every wavefront's share relative to the rows' common maximum, then the sum of the shares
        float2* const ml = (float2*)lds;
        if (quarter == 0)
#pragma unroll
            for (int nt = 0; nt < kNT; nt++) ml[wave * kRows + 16 * nt + n] = make_float2(m[nt], l[nt]);
        __syncthreads();
#pragma unroll
        for (int nt = 0; nt < kNT; nt++) {
            float top = -INFINITY, total = 0.f;
            for (int w = 0; w < waves; w++) top = fmaxf(top, ml[w * kRows + 16 * nt + n].x);
            const float ref = top == -INFINITY ? 0.f : top;
            for (int w = 0; w < waves; w++) total = fmaf(ml[w * kRows + 16 * nt + n].y, fast_exp2(ml[w * kRows + 16 * nt + n].x - ref), total);
            const float f = total > 0.f ? fast_exp2(m[nt] - ref) / total : 0.f;
#pragma unroll
            for (int cc = 0; cc < kC; cc++)
#pragma unroll
                for (int t = 0; t < 4; t++) o[cc][t][nt] *= f;
        }
        float4_t* const shares = (float4_t*)lds;  // (over the maxima, which every wavefront has read by then)
        constexpr int kRegs = kC * 4 * kNT;
        for (int half = waves >> 1; half > 0; half >>= 1) {
            __syncthreads();
            if (wave >= half && wave < 2 * half)
#pragma unroll
                for (int i = 0; i < kRegs; i++) shares[((wave - half) * kRegs + i) * 64 + lane] = o[i / (4 * kNT)][i / kNT % 4][i % kNT];
            __syncthreads();
            if (wave < half)
#pragma unroll
                for (int i = 0; i < kRegs; i++) o[i / (4 * kNT)][i / kNT % 4][i % kNT] += shares[(wave * kRegs + i) * 64 + lane];
        }
        if (wave != 0) return;
    } else {
#pragma unroll
        for (int nt = 0; nt < kNT; nt++) {
            const float f = l[nt] > 0.f ? 1.0f / l[nt] : 0.f;
#pragma unroll
            for (int cc = 0; cc < kC; cc++)
#pragma unroll
                for (int t = 0; t < 4; t++) o[cc][t][nt] *= f;
        }
    }
    // lane (row n, q): register e of o[cc][t] is column 64 cc + 16 q + 4 e + t, sixteen in a row
#pragma unroll
    for (int nt = 0; nt < kNT; nt++) {
        const int row = row0 + 16 * nt + n;
        // The products multiply masked keys by a zero probability (an infinite value row would make that NaN) and let
        // exponentials grow to 2^60 (times a value row above 1e20: infinity).  Rows that are not finite are worked again
        // the way that skips such keys and keeps its reference at the maximum; where the inputs do ask for it they stay so.
        float finite = 0.f;
#pragma unroll
        for (int cc = 0; cc < kC; cc++)
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (!kPad || 64 * cc + 16 * quarter + 4 * e < D) finite = fmaf(o[cc][t][nt][e], 0.f, finite);
        uint64_t bad = __builtin_amdgcn_ballot_w64(finite != 0.f && row < p.len_q);
        bad |= bad >> 32;
        bad = (bad | bad >> 16) & 0xffff;
        const bool again = (bad >> n) & 1;
        while (bad != 0) {
            const int r = row0 + 16 * nt + __builtin_ctzll(bad);
            bad &= bad - 1;
            const DenseKV kv{(const uint8_t*)k, (const uint8_t*)v, 4 * (int64_t)D, HIPATTN_F32};
            const float* const q_row = q + (int64_t)r * D;
            float x[kC];
            if constexpr (kForm == kNoMask) {
                attend_row_wave(q_row, kv, NoBias{}, 0, p.causal ? min(r + 1, p.len_kv) : p.len_kv, D, p.scale, x);
            } else {
                const int64_t at = (int64_t)b * p.mask_stride[0] + (int64_t)h * p.mask_stride[1] + (int64_t)r * p.mask_stride[2];
                const MaskRow bias{(const uint8_t*)p.mask + at * (p.mask_dtype == HIPATTN_U8 ? 1 : dtype_bytes(p.mask_dtype)),
                                   p.mask_stride[3], p.mask_dtype};
                attend_row_wave(q_row, kv, bias, 0, p.len_kv, D, p.scale, x);
            }
#pragma unroll
            for (int i = 0; i < kC; i++)
                if (lane + 64 * i < D) ((float*)p.out)[((int64_t)bh * p.len_q + r) * D + lane + 64 * i] = x[i];
        }
        if (row >= p.len_q || again) continue;
        float* const out = (float*)p.out + ((int64_t)bh * p.len_q + row) * D;
#pragma unroll
        for (int cc = 0; cc < kC; cc++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int d = 64 * cc + 16 * quarter + 4 * e;
                if (!kPad || d < D) *(float4_t*)(out + d) = (float4_t){o[cc][0][nt][e], o[cc][1][nt][e], o[cc][2][nt][e], o[cc][3][nt][e]};
            }
    }
}

template <int kDP, int kNT>
hipError_t launch(const SdpaParams& p, int waves, hipStream_t stream) {
    constexpr int kRows = 16 * kNT;
    const int q_tiles = (p.len_q + kRows - 1) / kRows;
    const int items = p.batch * p.num_heads_q * q_tiles;
    const size_t lds = waves > 1 ? (size_t)(waves / 2) * kRows * kDP * sizeof(float) : 0;  // (64 KB at most)
    const dim3 grid((unsigned)((items + 7) / 8 * 8)), block(64 * waves);
    const bool pad = p.head_dim < kDP;
    // causal: a head's longest query tiles first, so that short ones fill the end.  Where every wavefront is resident
    // from the start there is no end to fill: there the tiles of every other head go the other way, so that a
    // compute unit gets a long and a short one (16 heads of 2,048: 262 -> 202 us)
    const int snake = p.causal && (int64_t)items * waves <= 4096;
    const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, lds, stream, p, q_tiles, items, snake); };
    if (!p.mask)
        go(pad ? sdpa_f32_kernel<kDP, kNT, kNoMask, true> : sdpa_f32_kernel<kDP, kNT, kNoMask, false>);
    else if (p.mask_stride[3] == 1 && p.mask_dtype == HIPATTN_U8)
        go(pad ? sdpa_f32_kernel<kDP, kNT, kBoolean, true> : sdpa_f32_kernel<kDP, kNT, kBoolean, false>);
    else if (p.mask_stride[3] == 1 && p.mask_dtype == HIPATTN_F32)
        go(pad ? sdpa_f32_kernel<kDP, kNT, kFloat, true> : sdpa_f32_kernel<kDP, kNT, kFloat, false>);
    else
        go(pad ? sdpa_f32_kernel<kDP, kNT, kAnyMask, true> : sdpa_f32_kernel<kDP, kNT, kAnyMask, false>);
    return hipGetLastError();
}

}  // namespace

bool sdpa_f32_supported(const SdpaParams& p) {
    const auto aligned16 = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
    const int64_t tiles = (int64_t)p.batch * p.num_heads_q * ((p.len_q + 15) / 16);
    return p.dtype == HIPATTN_F32 && p.head_dim <= 128 && p.head_dim % 4 == 0 && p.len_kv > 0 && tiles < (1 << 30) && aligned16(p.q) &&
           aligned16(p.k) && aligned16(p.v) && aligned16(p.out);
}

// Row tiles per wavefront and wavefronts the keys are split over, from the time the busiest SIMD would take: the
// wavefronts it gets, times a wavefront's steps (the MFMAs' own cycles and the vector instructions beside them), plus
// what a wavefront costs however few its steps are (query rows, sharing out the result).  Measured around the lines it draws, with 1 / 2 / 4 / 8 wavefronts
// of one row tile: 8 heads of 128 rows, causal, size 64: 7.4 / 5.8 / 5.5 / 6.4 us; 12 heads of 475: 23.6 / 20.4 / 14.8 /
// 17.2; 2 x 16 heads of 512, causal, size 128: 38 / 28 / 42 / 45 (four do not fit beside each other); 7 x 8 heads of
// 164, causal, size 128: 15.5 / 13.4 / 15.9 / 22; 8 heads of 1,520, size 128: 113 / 108 / 104 / 112.  Two row tiles read K and V half as often per
// row: 2 x 8 heads of 2,048, size 64: 133 us with two wavefronts against 146 with one of one row tile; 5 x 12 heads of
// 897 rows and 132 keys, size 128: 47 against 53; under the causal flag they pay for twice the masked half of the
// diagonal (16 heads of 2,048, size 128: 193 against 164).
namespace {
struct Split {
    int row_tiles, waves;
};
Split choose_split(const SdpaParams& p) {
    const int64_t heads = (int64_t)p.batch * p.num_heads_q;
    const double mfma = p.head_dim <= 64 ? 1024 : 2048;  // cycles per step and row tile
    Split best{1, 1};
    double best_cost = 0;
    for (int nt = 1; nt <= (p.causal ? 1 : 2); nt++)
        for (int waves = 1; waves <= 8 && (waves == 1 || p.len_kv >= 16 * waves); waves *= 2) {
            const int64_t items = heads * ((p.len_q + 16 * nt - 1) / (16 * nt));
            const int64_t per_simd = (items * waves + 1023) / 1024;
            double steps = (p.len_kv + 15) / 16;
            if (p.causal && per_simd > 1) steps = (steps + 1) / 2;                 // (long and short ones mix)
            if (p.mask && p.mask_dtype == HIPATTN_U8) steps *= 0.75;               // (a padding mask leaves part of the keys)
            double cost = per_simd * (steps / waves * (nt * mfma + 110 + 30 * nt) + (waves == 1 ? 1500 : waves < 8 ? 3000 : 4500));
            const int resident = nt == 2 ? 2 : p.head_dim <= 64 ? 5 : 3;
            if (per_simd == 1) cost *= 1.3;                                        // (nobody to hide a wavefront's latencies)
            if (per_simd > resident) cost *= p.causal ? 1.5 : 1.2;                 // (the last ones start late)
            if (best_cost == 0 || cost < best_cost) best_cost = cost, best = {nt, waves};
        }
    return best;
}
}  // namespace

hipError_t launch_sdpa_f32(const SdpaParams& p, hipStream_t stream) {
    const Split s = choose_split(p);
    if (p.head_dim <= 64) return s.row_tiles == 1 ? launch<64, 1>(p, s.waves, stream) : launch<64, 2>(p, s.waves, stream);
    return s.row_tiles == 1 ? launch<128, 1>(p, s.waves, stream) : launch<128, 2>(p, s.waves, stream);
}

}  // namespace hipattn
