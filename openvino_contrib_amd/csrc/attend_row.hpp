// One query row by one wavefront in fp32 vector arithmetic: the row function of the shape-generic kernels, and what
// the fp32 matrix kernel falls back on for rows that come out infinite or not a number.
#pragma once

#include "device_common.hpp"

namespace hipattn {

constexpr int kGenericMaxD = 512;
constexpr int kGenericSlots = kGenericMaxD / 64;

// No additive term on the scores.
struct NoBias {
    __device__ __forceinline__ float operator()(int) const { return 0.0f; }
};

// ALiBi: slope * (key position - query position).
struct DistanceBias {
    float slope;
    int pos;
    __device__ __forceinline__ float operator()(int j) const { return slope * (float)(j - pos); }
};

// One row of an attention mask: element j at row + j * stride (stride 0: broadcast over the keys).
// Boolean masks (u8, nonzero = the key takes part) become 0 / -inf; float masks are added to the
// scaled scores, as ScaledDotProductAttention specifies.
struct MaskRow {
    const uint8_t* row;
    int64_t stride;  // elements
    int dtype;       // HIPATTN_F32 / F16 / BF16, or HIPATTN_U8 for boolean
    __device__ __forceinline__ float operator()(int j) const {
        if (dtype == HIPATTN_U8) return row[j * stride] ? 0.0f : -INFINITY;
        return load_scalar(row, j * stride, dtype);
    }
};

// Attend one query row to keys [j0, j1).  q_row is the row in fp32 (LDS or global memory); KV yields row
// pointers and says which keys exist (a key in a block outside the cache has probability zero);
// bias(j) is added to the scaled score of key j.  Every lane of the wavefront must call this; the
// result for head-dim slot d = lane + 64 * i < 64 * kSlots is returned in o[i], already normalised.  A row that
// can attend nothing (empty range, every key masked with -inf) yields zeros.
// sink: -INFINITY, or a logit that joins the row's softmax without a value row (the denominator grows by exp(sink)).
template <int kSlots, typename KV, typename Bias>
__device__ __forceinline__ void attend_row_wave(const float* q_row, const KV& kv, const Bias& bias, int j0, int j1, int D,
                                                float scale, float (&o)[kSlots], float sink = -INFINITY) {
    const int lane = threadIdx.x & 63;
    float m = -INFINITY, l = 0.0f;
#pragma unroll
    for (int i = 0; i < kSlots; i++) o[i] = 0.0f;
    const float c = scale * kLog2e;
    for (int base = j0; base < j1; base += 64) {
        const int j = base + lane;
        float s = -INFINITY;
        if (j < j1 && kv.exists(j)) {
            const uint8_t* krow = kv.k_row(j);
            float acc = 0.0f;
            for (int d = 0; d < D; d++) acc = fmaf(q_row[d], load_cache_elem(krow, d, kv.dtype), acc);
            s = fmaf(acc, c, bias(j) * kLog2e);
        }
        const float m_new = fmaxf(m, wave_max(s));
        if (m_new == -INFINITY) continue;  // nothing attended so far (wave-uniform)
        const float alpha = fast_exp2(m - m_new);  // exp2(-inf) = 0 on the first tile
        const float pj = (s != -INFINITY) ? fast_exp2(s - m_new) : 0.0f;
        l = l * alpha + wave_sum(pj);
        m = m_new;
#pragma unroll
        for (int i = 0; i < kSlots; i++) o[i] *= alpha;
        const int n = min(64, j1 - base);
        for (int jj = 0; jj < n; jj++) {
            const float pb = __shfl(pj, jj, 64);
            if (pb == 0.0f) continue;  // (wave-uniform) masked keys may be unreadable or hold anything
            const uint8_t* vrow = kv.v_row(base + jj);
#pragma unroll
            for (int i = 0; i < kSlots; i++) {
                const int d = lane + 64 * i;
                if (d < D) o[i] = fmaf(pb, load_cache_elem(vrow, d, kv.dtype), o[i]);
            }
        }
    }
    if (l > 0.0f && sink != -INFINITY) l += fast_exp2(sink * kLog2e - m);
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int i = 0; i < kSlots; i++) o[i] *= inv;
}

struct DenseKV {
    const uint8_t* k;
    const uint8_t* v;
    int64_t row_bytes;
    int dtype;
    __device__ __forceinline__ bool exists(int) const { return true; }
    __device__ __forceinline__ const uint8_t* k_row(int j) const { return k + j * row_bytes; }
    __device__ __forceinline__ const uint8_t* v_row(int j) const { return v + j * row_bytes; }
};

}  // namespace hipattn
