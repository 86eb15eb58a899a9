// The kernels and launches of the paged-attention fast path: schedule and cache write (prologue), decode (the loop is that of
// paged_decode.hpp, up to head size 128; head sizes above 128 here), merge, and where the chunks of a mixed batch run.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "paged_decode.hpp"

namespace hipattn {

// ---- plan ----------------------------------------------------------------------------------
// Exclusive prefix sums over the sequences of (a) attended blocks of decode sequences and
// (b) 128-row query tiles of multi-token sequences.  One workgroup; sequences are split evenly
// over the threads.
__device__ __forceinline__ void plan_block(const PagedParams& p) {
    __shared__ int wave_blk[4];
    __shared__ int wave_tile[4];
    __shared__ float wave_keys[4];
    const int tid = threadIdx.x;
    if (tid < 64) p.dyn_counter[tid] = 0;  // tickets for the dynamic pieces of this call, one counter per group
    const int per = (p.num_rows + 255) / 256;
    const int s0 = min(tid * per, p.num_rows), s1 = min(s0 + per, p.num_rows);
    const int tiled = p.lone_tile ? 1 : 2;  // tokens of the shortest sequence that gets query tiles
    int blk = 0, tile = 0;
    float key_tiles = 0.0f;  // 64-key tiles the flash kernel works through, summed over 128-row query tiles
    for (int s = s0; s < s1; s++) {
        // (rows are sequences whenever the lengths matter here: max_q_tiles > 0)
        const int qlen = p.max_q_tiles > 0 ? p.subsequence_begins[s + 1] - p.subsequence_begins[s] : 1;
        if (!p.lone_tile) blk += line_units(decode_range(p, s).nb, p.switch_cost);
        tile += (qlen >= tiled && p.max_q_tiles > 0) ? (qlen + 127) / 128 : 0;
        if (p.overlap && qlen >= tiled) {
            const int past = p.past_lens[s];
            for (int r0 = 0; r0 < qlen; r0 += 128) {
                int keys = past + min(qlen, r0 + 128);
                if (p.sliding_window > 0) keys = min(keys, p.sliding_window + 128);
                key_tiles += (float)((keys + 63) >> 6);
            }
        }
    }
    // Exclusive prefix sums over the 256 threads: a scan inside each wavefront (six shuffle steps),
    // then the totals of the wavefronts ahead.  (One thread adding up 256 values in LDS took about as
    // long as the rest of the launch.)
    const int lane = tid & 63, wv = tid >> 6;
    int scan_blk = blk, scan_tile = tile;
    float scan_keys = key_tiles;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int ub = __shfl_up(scan_blk, d, 64), ut = __shfl_up(scan_tile, d, 64);
        const float uk = __shfl_up(scan_keys, d, 64);
        if (lane >= d) {
            scan_blk += ub;
            scan_tile += ut;
            scan_keys += uk;
        }
    }
    if (lane == 63) {
        wave_blk[wv] = scan_blk;
        wave_tile[wv] = scan_tile;
        wave_keys[wv] = scan_keys;
    }
    __syncthreads();
    int ahead_blk = 0, ahead_tile = 0, total_blk = 0;
    float total_keys = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        ahead_blk += w < wv ? wave_blk[w] : 0;
        ahead_tile += w < wv ? wave_tile[w] : 0;
        total_blk += wave_blk[w];
        total_keys += wave_keys[w];
    }
    if (tid == 0 && p.overlap) {
        // Compute-unit time of the two parts, in microseconds, as measured with both running:
        // a compute unit of the decode kernel streams about 33 GB/s of fp16 cache (u8: 24 GB/s),
        // one of the flash kernel does a 128-row x 64-key tile of one head in about 1.1 us
        // (u8 caches, dequantised on the way: 1.4 us).  Each part gets compute units in
        // proportion to its work, so that both end together.
        const bool u8 = p.cache_dtype == HIPATTN_U8;
        const float decode_us = (float)total_blk * p.num_heads_kv * (u8 ? 8704.0f / 24000.0f : 16384.0f / 33000.0f) * p.overlap_share;
        const float prefill_us = total_keys * p.num_heads_q * (u8 ? 1.4f : 1.1f);
        const int cus = p.num_waves >> 3;
        int mine = (int)ceilf(cus * decode_us / fmaxf(decode_us + prefill_us, 1.0f));
        mine = max(1, min(mine, cus));
        p.plan_waves[0] = mine * 8;
    }
    blk = ahead_blk + scan_blk - blk;
    tile = ahead_tile + scan_tile - tile;
    for (int s = s0; s < s1; s++) {
        const int qlen = p.max_q_tiles > 0 ? p.subsequence_begins[s + 1] - p.subsequence_begins[s] : 1;
        p.blk_prefix[s] = blk;
        p.tile_prefix[s] = tile;
        DecodeRange rg = decode_range(p, s);
        if (p.lone_tile) rg.nb = 0, rg.empty_row = 0;
        ((DecodeRange*)p.seq_info)[s] = rg;
        if (rg.empty_row) zero_output_row(p, rg.token);  // (rare: an empty block table) nothing will visit this row
        blk += line_units(rg.nb, p.switch_cost);
        tile += (qlen >= tiled && p.max_q_tiles > 0) ? (qlen + 127) / 128 : 0;
    }
    if (s1 == p.num_rows && s0 < p.num_rows) {
        p.blk_prefix[p.num_rows] = blk;
        p.tile_prefix[p.num_rows] = tile;
    }
}

// One launch for step 1 of the operator and the schedule: workgroups [0, write_blocks) scatter
// the new K/V rows into the caches (four wavefronts of the writer each), workgroup write_blocks
// plans.  The plan reads lengths only, never the cache, so the two parts do not interact.
__global__ __launch_bounds__(256) void paged_prologue_kernel(KvWriteParams wp, PagedParams p, int write_blocks) {
    if ((int)blockIdx.x < write_blocks) {
        const int64_t wv = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
        if (wp.head_dim <= 128)  // (elements of a row per lane: two up to head size 128, four up to 256)
            kv_cache_write_wave<2>(wp, wv, threadIdx.x & 63);
        else
            kv_cache_write_wave<4>(wp, wv, threadIdx.x & 63);
    } else {
        plan_block(p);
    }
}

// Log-sum-exp reduction of the partials that pieces id_first..id_last left for query head g of
// segment (s, h), done by kParts wavefronts of a workgroup, of which `part` takes every kParts-th piece (their
// sums meet in LDS).  Pieces are taken 64 at a time: lane i fetches the (max, sum) pair of piece i, the weights
// come out of two wavefront reductions, and the output rows are then accumulated eight pieces at a time, the
// eight loads ahead of the first use (lane l owns head-dim 2l and 2l + 1 and, at head size 256, 128 + 2l, 129 + 2l).
template <int kParts>
__device__ __forceinline__ void merge_segment_head(const PagedParams& p, const Line& line, int s, int h, int g,
                                                   int token, int id_first, int id_last, int part, int lane,
                                                   float4 (*shares)[64]) {
    const int Hkv = p.num_heads_kv, G = p.num_heads_q / p.num_heads_kv, D = p.head_dim;
    const int64_t seg_slot = (int64_t)s * Hkv + h;
    const bool all_live = line.P == 0 && line.total >= line.W;  // no piece of the line is empty
    const auto live = [&](int id) { return id <= id_last && (all_live || line.begin(id) < line.begin(id + 1)); };
    float m_run = -INFINITY, l_run = 0.0f, ox[2] = {0.0f, 0.0f}, oy[2] = {0.0f, 0.0f};
    for (int id0 = id_first; id0 <= id_last; id0 += 64) {
        const bool have = live(id0 + lane);  // (empty pieces leave nothing)
        float mw = -INFINITY, lw = 0.0f;
        if (have) {
            const float2 ml = *(const float2*)(p.part_ml + ((seg_slot + id0 + lane) * G + g) * 2);
            mw = ml.x;
            lw = ml.y;
        }
        const uint64_t alive = __builtin_amdgcn_ballot_w64(have);
        const float m_new = fmaxf(m_run, wave_max(mw));
        const float rescale = (m_run == -INFINITY) ? 0.0f : fast_exp2(m_run - m_new);
        const float f = (mw == -INFINITY) ? 0.0f : fast_exp2(mw - m_new);
        l_run = l_run * rescale + wave_sum(f * lw);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            ox[c] *= rescale;
            oy[c] *= rescale;
        }
        m_run = m_new;
        const int n = min(64, id_last - id0 + 1);
        const auto rows = [&](int c) __attribute__((always_inline)) {
            const int d = 128 * c + 2 * lane;
            const float* const at = p.part_out + ((seg_slot + id0) * G + g) * D + (d < D ? d : 0);
            for (int i0 = part; i0 < n; i0 += 8 * kParts) {
                float2 v[8];
                float fi[8];
#pragma unroll
                for (int u = 0; u < 8; u++) {  // (a piece that does not exist: zeros with weight zero)
                    const int i = i0 + u * kParts;
                    const bool ok = i < n && ((alive >> i) & 1) != 0;
                    fi[u] = ok ? __shfl(f, i, 64) : 0.0f;
                    v[u] = ok ? *(const float2*)(at + (int64_t)i * G * D) : make_float2(0.0f, 0.0f);
                }
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    ox[c] = fmaf(fi[u], v[u].x, ox[c]);
                    oy[c] = fmaf(fi[u], v[u].y, oy[c]);
                }
            }
        };
        rows(0);
        if (D > 128) rows(1);
    }
    if constexpr (kParts > 1) {
        if (part > 0) shares[part - 1][lane] = make_float4(ox[0], oy[0], ox[1], oy[1]);
        __syncthreads();
        if (part > 0) return;
#pragma unroll
        for (int i = 0; i < kParts - 1; i++) {
            const float4 v = shares[i][lane];
            ox[0] += v.x, oy[0] += v.y, ox[1] += v.z, oy[1] += v.w;
        }
    }
    // (the attention sink of the head, when there is one: a logit in the denominator without a value row)
    if (p.sinks != nullptr && l_run > 0.0f) l_run += fast_exp2(p.sinks[h * G + g] * kLog2e - m_run);
    const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int d = 128 * c + 2 * lane;
        if (d >= D) continue;
        const int64_t o = ((int64_t)token * p.num_heads_q + (int64_t)h * G + g) * D + d;
        if (p.out_dtype == HIPATTN_F32) {
            *(float2*)((float*)p.out + o) = make_float2(ox[c] * inv, oy[c] * inv);
        } else {
            const uint32_t lo = p.out_dtype == HIPATTN_F16 ? float_to_f16_bits(ox[c] * inv) : float_to_bf16_bits(ox[c] * inv);
            const uint32_t hi = p.out_dtype == HIPATTN_F16 ? float_to_f16_bits(oy[c] * inv) : float_to_bf16_bits(oy[c] * inv);
            *(uint32_t*)((uint16_t*)p.out + o) = lo | (hi << 16);
        }
    }
}

template <bool kU8, bool kBf16, int kWaves, bool kSelfPlan = false, int kHD = kD, int kBlk = kBS, bool kPad = false, bool kAlibi = false, bool kHalfFromBf16 = false>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void paged_decode_kernel(PagedParams p, KvWriteParams wp, int do_write) {
    paged_decode_body<kU8, kBf16, kWaves, kSelfPlan, kHD, kBlk, kPad, kAlibi, kHalfFromBf16>(p, wp, do_write, (int)blockIdx.x);
}

// ---- head size 256 ------------------------------------------------------------------------------
// The same schedule, products and lane layouts, with the head dimension worked through in two
// halves of 128 columns so that the registers hold: a unit of 32 tokens arrives as four
// half-stages of 32 registers -- K columns 0..127, K columns 128..255, V columns 0..127, V columns
// 128..255 -- the scores are the sum of the two K halves' products, the probabilities go into two
// sets of output accumulators, and while one half-stage is consumed the next is in flight.  A
// wavefront therefore has half as many bytes in flight as the head-128 kernel, and twice as many
// wavefronts are launched (eight per compute unit).
struct HalfRegs {
    uint4_t x[8];  // K: [tile * 4 + piece]; V: [tile * 4 + row]
};

// row: bytes from one cache row to the next (512, or 2 * head_dim for a smaller head).  koff[i]: this
// lane's offset of K piece i of the half inside a tile (a piece past the end of the row is pointed at
// the row's first piece: valid memory that meets zeros in the query operand).
template <int kBlk>
__device__ __forceinline__ void load_k_half(HalfRegs& b, const uint8_t* const (&kb)[2], int row, const int (&koff)[4]) {
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint8_t* const kt = kBlk == 32 ? kb[0] + t * 16 * row : kb[t];
#pragma unroll
        for (int i = 0; i < 4; i++) b.x[t * 4 + i] = *(const uint4_t*)(kt + koff[i]);
    }
}

// voff: this lane's offset of its first V row's piece of the half; v_ok: its columns exist.
template <int kBlk>
__device__ __forceinline__ void load_v_half(HalfRegs& b, const uint8_t* const (&vb)[2], int row, int voff, bool v_ok) {
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint8_t* const vt = kBlk == 32 ? vb[0] + t * 16 * row : vb[t];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            uint4_t piece = {0u, 0u, 0u, 0u};
            if (v_ok) piece = *(const uint4_t*)(vt + voff + r * row);
            b.x[t * 4 + r] = piece;
        }
    }
}

struct WaveState256 {
    float m, l;
    float corr;  // u8 only: this lane's share of sum_j p'_j (zp_j + bias)
    float4_t acc[2][8];  // acc[half][e][r] = O[head][128 * half + (kg*4 + r)*8 + e]
};

template <bool kBf16>
__device__ __forceinline__ void scores_half(float4_t (&s)[2], const HalfRegs& k, const typename Op16<kBf16>::vec8 (&q)[4]) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) s[t] = Op16<kBf16>::mma(Op16<kBf16>::from_bits(k.x[t * 4 + i]), q[i], s[t]);
}

// Mask, scale and online softmax of a unit's scores (lane: tokens tok_base + t*16 + kg*4 + r); the
// accumulators are rescaled when a row's maximum moved.  Returns the probabilities as the B operand.
template <bool kBf16>
__device__ __forceinline__ typename Op16<kBf16>::vec8 softmax_unit(WaveState256& st, const float4_t (&s)[2], float c, int tok_base,
                                                                  int j0, int ctx, int kg, int tiles) {
    float sv[8];
    float mloc = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int tok = tok_base + t * 16 + kg * 4 + r;
            const float x = (tok >= j0 && tok < ctx && ((tiles >> t) & 1)) ? s[t][r] * c : -INFINITY;
            sv[t * 4 + r] = x;
            mloc = fmaxf(mloc, x);
        }
    mloc = max_over_rows(mloc);
    const float m_new = fmaxf(st.m, mloc);
    // (-inf only while nothing has been attended yet and this unit's blocks both lie outside the cache:
    // everything stays at zero then; exp2(-inf - -inf) would be NaN)
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    const float alpha = fast_exp2(st.m - m_use);
    st.m = m_new;
    typename Op16<kBf16>::vec8 pf;
    float lsum = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const float pj = fast_exp2(sv[j] - m_use);
        lsum += pj;
        Op16<kBf16>::set(pf, j, pj);
    }
    st.l = st.l * alpha + lsum;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int e = 0; e < 8; e++) st.acc[h][e] *= alpha;
    }
    return pf;
}

// O^T += V^T P^T for one half of the columns.  Rows outside the attended range may hold anything
// (never-written cache memory): their probability is exactly zero and they are cleared, so that
// 0 * NaN cannot occur.
template <bool kBf16>
__device__ __forceinline__ void pv_half(float4_t (&acc)[8], HalfRegs& v, typename Op16<kBf16>::vec8 pf, bool partial, int tok_base,
                                        int j0, int ctx, int kg, int tiles) {
    if (partial) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int tok = tok_base + (j >> 2) * 16 + kg * 4 + (j & 3);
            if (!(tok >= j0 && tok < ctx && ((tiles >> (j >> 2)) & 1))) v.x[j] = (uint4_t){0u, 0u, 0u, 0u};
        }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) {
        uint4_t w;
#pragma unroll
        for (int jp = 0; jp < 4; jp++) {
            const uint32_t lo = v.x[2 * jp][e >> 1], hi = v.x[2 * jp + 1][e >> 1];
            w[jp] = (e & 1) ? pack_hi(lo, hi) : pack_lo(lo, hi);
        }
        acc[e] = Op16<kBf16>::mma(Op16<kBf16>::from_bits(w), pf, acc[e]);
    }
}

// ---- the same for u8 caches: a half-stage is 32 tokens x 128 bytes (16 registers), so K (both halves, plus
// the tokens' scales and zero-points) and V (both halves) are the two stages that alternate, and a
// wavefront has as many bytes in flight as with a 16-bit cache.
struct HalfRegs8 {
    uint2_t x[8];  // K: [tile * 4 + piece]; V: [tile * 4 + row]
};

template <int kBlk>
__device__ __forceinline__ void load_k_half8(HalfRegs8& b, const uint8_t* const (&kb)[2], int row, const int (&koff)[4]) {
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint8_t* const kt = kBlk == 32 ? kb[0] + t * 16 * row : kb[t];
#pragma unroll
        for (int i = 0; i < 4; i++) b.x[t * 4 + i] = *(const uint2_t*)(kt + koff[i]);
    }
}

template <int kBlk>
__device__ __forceinline__ void load_v_half8(HalfRegs8& b, const uint8_t* const (&vb)[2], int row, int voff, bool v_ok) {
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint8_t* const vt = kBlk == 32 ? vb[0] + t * 16 * row : vb[t];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            uint2_t piece = {0u, 0u};
            if (v_ok) piece = *(const uint2_t*)(vt + voff + r * row);
            b.x[t * 4 + r] = piece;
        }
    }
}

// (scale, zp) of one token per lane, laid out as in BlockRegs<true>
template <int kBlk>
__device__ __forceinline__ float2 load_scale_zp(const uint8_t* const (&kb)[2], const uint8_t* const (&vb)[2], int row, int n16, int kg) {
    const int j = n16 & 7, at = (kg * 4 + (j & 3)) * row;
    if constexpr (kBlk == 32) {
        return *(const float2*)((n16 < 8 ? kb[0] : vb[0]) + (j >> 2) * 16 * row + at);
    } else {  // (one of four tile bases per lane, put together arithmetically: see load_block)
        const uintptr_t k0 = (uintptr_t)kb[0], k1 = (uintptr_t)kb[1], v0 = (uintptr_t)vb[0], v1 = (uintptr_t)vb[1];
        const uintptr_t second = (uintptr_t)(j >> 2), value = (uintptr_t)(n16 >> 3);
        const uintptr_t in_k = k0 + second * (k1 - k0), in_v = v0 + second * (v1 - v0);
        return *(const float2*)(in_k + value * (in_v - in_k) + (uintptr_t)at);
    }
}

__device__ __forceinline__ void scores_half8(float4_t (&s)[2], const HalfRegs8& k, const Op16<false>::vec8 (&q)[4]) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint4_t w;
            w[0] = bytes_to_biased_half2(k.x[t * 4 + i][0], 0x04010400u);
            w[1] = bytes_to_biased_half2(k.x[t * 4 + i][0], 0x04030402u);
            w[2] = bytes_to_biased_half2(k.x[t * 4 + i][1], 0x04010400u);
            w[3] = bytes_to_biased_half2(k.x[t * 4 + i][1], 0x04030402u);
            s[t] = Op16<false>::mma(Op16<false>::from_bits(w), q[i], s[t]);
        }
}

// softmax_unit for byte scores: the tokens' scales and zero-points turn them into scores, the
// probabilities leave multiplied by V's scales, and st.corr collects sum_j p'_j (zp_j + bias).
__device__ __forceinline__ Op16<false>::vec8 softmax_unit8(WaveState256& st, const float4_t (&s)[2], float2 sz, float sumq, float c,
                                                          int tok_base, int j0, int ctx, int kg, int tiles, bool partial) {
    float sz_scale = sz.x, sz_zero = sz.y + kByteBias;
    if (partial) {  // rows outside the attended range may hold anything: their scale and zero-point are cleared
        const int j = ((int)threadIdx.x & 7), tok = tok_base + (j >> 2) * 16 + kg * 4 + (j & 3);
        if (!(tok >= j0 && tok < ctx && ((tiles >> (j >> 2)) & 1))) sz_scale = sz_zero = 0.0f;
    }
    const float sz_prod = sz_scale * sz_zero;
    float ks[8], kp[8], vs[8], vz[8];
    ks[0] = row_broadcast<0>(sz_scale); kp[0] = row_broadcast<0>(sz_prod); vs[0] = row_broadcast<8>(sz_scale); vz[0] = row_broadcast<8>(sz_zero);
    ks[1] = row_broadcast<1>(sz_scale); kp[1] = row_broadcast<1>(sz_prod); vs[1] = row_broadcast<9>(sz_scale); vz[1] = row_broadcast<9>(sz_zero);
    ks[2] = row_broadcast<2>(sz_scale); kp[2] = row_broadcast<2>(sz_prod); vs[2] = row_broadcast<10>(sz_scale); vz[2] = row_broadcast<10>(sz_zero);
    ks[3] = row_broadcast<3>(sz_scale); kp[3] = row_broadcast<3>(sz_prod); vs[3] = row_broadcast<11>(sz_scale); vz[3] = row_broadcast<11>(sz_zero);
    ks[4] = row_broadcast<4>(sz_scale); kp[4] = row_broadcast<4>(sz_prod); vs[4] = row_broadcast<12>(sz_scale); vz[4] = row_broadcast<12>(sz_zero);
    ks[5] = row_broadcast<5>(sz_scale); kp[5] = row_broadcast<5>(sz_prod); vs[5] = row_broadcast<13>(sz_scale); vz[5] = row_broadcast<13>(sz_zero);
    ks[6] = row_broadcast<6>(sz_scale); kp[6] = row_broadcast<6>(sz_prod); vs[6] = row_broadcast<14>(sz_scale); vz[6] = row_broadcast<14>(sz_zero);
    ks[7] = row_broadcast<7>(sz_scale); kp[7] = row_broadcast<7>(sz_prod); vs[7] = row_broadcast<15>(sz_scale); vz[7] = row_broadcast<15>(sz_zero);
    float sv[8];
    float mloc = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = t * 4 + r, tok = tok_base + t * 16 + kg * 4 + r;
            const float x = fmaf(ks[j], s[t][r], -(kp[j] * sumq));
            sv[j] = (tok >= j0 && tok < ctx && ((tiles >> t) & 1)) ? x * c : -INFINITY;
            mloc = fmaxf(mloc, sv[j]);
        }
    mloc = max_over_rows(mloc);
    const float m_new = fmaxf(st.m, mloc);
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;  // (see softmax_unit)
    const float alpha = fast_exp2(st.m - m_use);
    st.m = m_new;
    Op16<false>::vec8 pf;
    float lsum = 0.0f, csum = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        float pj = fast_exp2(sv[j] - m_use);
        lsum += pj;
        pj *= vs[j];
        Op16<false>::set(pf, j, pj);
        csum = fmaf(Op16<false>::get(pf, j), vz[j], csum);
    }
    st.l = st.l * alpha + lsum;
    st.corr = st.corr * alpha + csum;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int e = 0; e < 8; e++) st.acc[h][e] *= alpha;
    }
    return pf;
}

// O^T += V^T P^T for one half of the columns, V as biased bytes (every byte is a finite number, and
// the probabilities of rows outside the attended range are exactly zero)
__device__ __forceinline__ void pv_half8(float4_t (&acc)[8], const HalfRegs8& v, Op16<false>::vec8 pf) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
        uint4_t w;
        const uint32_t sel = 0x0c000c00u | ((4u + (e & 3)) << 16) | (uint32_t)(e & 3);
#pragma unroll
        for (int jp = 0; jp < 4; jp++) w[jp] = bytes_to_biased_half2(v.x[2 * jp][e >> 2], v.x[2 * jp + 1][e >> 2], sel);
        acc[e] = Op16<false>::mma(Op16<false>::from_bits(w), pf, acc[e]);
    }
}

// kPad: the call's head size (p.head_dim, a multiple of 8 above 128) may be smaller than 256.
// kU8: a u8 cache (fp16 operands).
template <bool kBf16, int kBlk, bool kPad, bool kU8 = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) void paged_decode256_kernel(PagedParams p) {
    static_assert(!(kU8 && kBf16), "u8 caches are dequantised to fp16 operands");
    // kBlk: 16, 32, or 0 for any larger power of two (p.block_size: a block then holds several units)
    constexpr int kEntries = kBlk == 16 ? 2 : 1;
    constexpr int kTileBlk = kBlk == 16 ? 16 : 32;
    const int blk = kBlk ? kBlk : p.block_size;
    const int sub_mask = kBlk ? 0 : (p.block_size >> 5) - 1;
    const int sub_shift = kBlk ? 0 : __builtin_ctz(p.block_size >> 5);
    const int w = blockIdx.x, lane = threadIdx.x, n16 = lane & 15, kg = lane >> 4;
    const int kHD = kPad ? p.head_dim : 256;  // (a constant unless kPad)
    const int kRowBytes = kU8 ? kHD + 8 : 2 * kHD;
    // this lane's piece offsets inside a tile, per half, and whether its V columns exist
    int koff[2][4], voff[2];
    bool v_ok[2];
#pragma unroll
    for (int half = 0; half < 2; half++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int first = half * 128 + kg * 32 + i * 8;  // first of the piece's eight columns
            koff[half][i] = n16 * kRowBytes + (kU8 ? 8 + (first < kHD ? first : 0) : (first < kHD ? first * 2 : 0));
        }
        voff[half] = kg * 4 * kRowBytes + (kU8 ? 8 + half * 128 + n16 * 8 : half * 256 + n16 * 16);
        v_ok[half] = half * 128 + n16 * 8 < kHD;
    }
    const int Hkv = p.num_heads_kv, G = p.num_heads_q / p.num_heads_kv;
    const float c = p.scale * kLog2e;
    const int64_t total = (int64_t)p.blk_prefix[p.num_rows] * Hkv;
    if (total <= 0) return;
    const int num_waves = working_waves(p, total, p.num_waves);
    if (w >= num_waves) return;
    const Line line(total, num_waves, 0);
    const int64_t block_stride = (int64_t)(Hkv / p.kv_share) * blk * kRowBytes;
    int64_t L = line.begin(w);
    const int64_t L_end = line.begin(w + 1);
    if (L >= L_end) return;
    int s = locate_sequence(p.blk_prefix, p.num_rows, (int)(L / Hkv), lane);
    while (L < L_end) {
        while (s + 1 < p.num_rows && (int64_t)p.blk_prefix[s + 1] * Hkv <= L) s++;  // next row with units
        const DecodeRange rg = ((const DecodeRange*)p.seq_info)[s];
        const int nb = rg.nb;
        if (nb <= 0) break;  // cannot happen for a consistent plan; never loop forever
        const int seglen = nb + p.switch_cost;
        const int64_t seq_L0 = (int64_t)p.blk_prefix[s] * Hkv;
        const int h = (int)((L - seq_L0) / seglen);
        const int64_t seg_B0 = seq_L0 + (int64_t)h * seglen + p.switch_cost;
        const int64_t seg_L1 = seg_B0 + nb;
        const int64_t from = max(L, seg_B0), to = min(L_end, seg_L1);
        if (from >= to) {
            L = to;
            continue;
        }
        const int b_rel = (int)(from - seg_B0);
        const int n = (int)(to - from);
        const bool whole = (n == nb);
        L = from;
        const int lb0 = rg.j0 / kUnit + b_rel;
        const int32_t* table = p.block_indices + rg.table_begin + (kBlk ? lb0 * kEntries : 0);
        const int entries = (rg.ctx + blk - 1) / blk - (kBlk ? lb0 * kEntries : 0);
        const int64_t head_off = (int64_t)(p.kv_share == 1 ? h : h / p.kv_share) * blk * kRowBytes;

        // Q^T operand in two halves: lane (head n16, kg) holds Q[head][128*half + kg*32 + i*8 .. +8]
        typename Op16<kBf16>::vec8 qf[2][4];
        float sumq = 0.0f;  // u8: the sum of the head's query elements (see process_block)
        {
            const int64_t qrow = ((int64_t)rg.token * p.num_heads_q + (int64_t)h * G + n16) * kHD;
#pragma unroll
            for (int half = 0; half < 2; half++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (n16 < G && half * 128 + kg * 32 + i * 8 < kHD) {
                        qf[half][i] = load_q8<kBf16>(p.q, qrow + half * 128 + kg * 32 + i * 8, p.q_dtype);
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; e++) Op16<kBf16>::set(qf[half][i], e, 0.0f);
                    }
                    if constexpr (kU8) {
#pragma unroll
                        for (int e = 0; e < 8; e++) sumq += Op16<kBf16>::get(qf[half][i], e);
                    }
                }
            if constexpr (kU8) {
                sumq += __shfl_xor(sumq, 16, 64);
                sumq += __shfl_xor(sumq, 32, 64);
            }
        }
        WaveState256 st;
        st.m = -INFINITY;
        st.l = 0.0f;
        st.corr = 0.0f;
#pragma unroll
        for (int half = 0; half < 2; half++)
#pragma unroll
            for (int e = 0; e < 8; e++) st.acc[half][e] = (float4_t){0.f, 0.f, 0.f, 0.f};

        constexpr int kGroup = 64 / kEntries;
        for (int g0 = 0; g0 < n; g0 += kGroup) {
            const int gn = min(kGroup, n - g0);
            const int my_entry = kBlk ? g0 * kEntries + lane : (lb0 + g0 + lane) >> sub_shift;
            const int my_pb = (lane < gn * kEntries && my_entry < entries) ? table[my_entry] : -1;
            // Bases of the two tiles of unit i, and which of them lie in a block of the cache.  A block id
            // outside the cache is replaced by one inside it, so that the loads need no branch; the mask
            // keeps such a tile out of the scores and clears its V rows.
            auto unit = [&](int i, const uint8_t* (&kb)[2], const uint8_t* (&vb)[2]) -> int {
                if constexpr (kEntries == 1) {
                    const int pb = __builtin_amdgcn_readlane(my_pb, i);
                    const int ok = (pb >= 0 && pb < p.num_blocks) ? 3 : 0;
                    int64_t off = (int64_t)min(max(pb, 0), p.num_blocks - 1) * block_stride + head_off;
                    if constexpr (kBlk == 0) off += (int64_t)((lb0 + g0 + i) & sub_mask) * (kUnit * kRowBytes);
                    kb[0] = p.key_cache + off;
                    kb[1] = kb[0] + 16 * kRowBytes;
                    vb[0] = p.value_cache + off;
                    vb[1] = vb[0] + 16 * kRowBytes;
                    return ok;
                } else {
                    const int pb0 = __builtin_amdgcn_readlane(my_pb, 2 * i), pb1 = __builtin_amdgcn_readlane(my_pb, 2 * i + 1);
                    const int ok = (pb0 >= 0 && pb0 < p.num_blocks ? 1 : 0) | (pb1 >= 0 && pb1 < p.num_blocks ? 2 : 0);
                    const int64_t off0 = (int64_t)min(max(pb0, 0), p.num_blocks - 1) * block_stride + head_off;
                    const int64_t off1 = (int64_t)min(max(pb1, 0), p.num_blocks - 1) * block_stride + head_off;
                    kb[0] = p.key_cache + off0;
                    kb[1] = p.key_cache + off1;
                    vb[0] = p.value_cache + off0;
                    vb[1] = p.value_cache + off1;
                    return ok;
                }
            };
            if constexpr (kU8) {
                // Two stages: K of unit i (both halves, with the scales and zero-points) is there when
                // iteration i begins; V arrives while the scores are worked out, the next unit's K while
                // the outputs are.  No branch in the body, as below.
                HalfRegs8 rk[2], rv[2];
                float2 sz;
                {
                    const uint8_t *kb[2], *vb[2];
                    (void)unit(0, kb, vb);
                    load_k_half8<kTileBlk>(rk[0], kb, kRowBytes, koff[0]);
                    load_k_half8<kTileBlk>(rk[1], kb, kRowBytes, koff[1]);
                    sz = load_scale_zp<kTileBlk>(kb, vb, kRowBytes, n16, kg);
                }
                for (int i = 0; i < gn; i++) {
                    const int tok_base = (lb0 + g0 + i) * kUnit;
                    const uint8_t *kb[2], *vb[2];
                    const int ok = unit(i, kb, vb);
                    const bool partial = (tok_base < rg.j0) || (tok_base + kUnit > rg.ctx) || ok != 3;  // wavefront-uniform
                    float4_t sc[2] = {(float4_t){0.f, 0.f, 0.f, 0.f}, (float4_t){0.f, 0.f, 0.f, 0.f}};
                    load_v_half8<kTileBlk>(rv[0], vb, kRowBytes, voff[0], v_ok[0]);
                    load_v_half8<kTileBlk>(rv[1], vb, kRowBytes, voff[1], v_ok[1]);
                    scores_half8(sc, rk[0], qf[0]);
                    scores_half8(sc, rk[1], qf[1]);
                    const Op16<false>::vec8 pf = softmax_unit8(st, sc, sz, sumq, c, tok_base, rg.j0, rg.ctx, kg, ok, partial);
                    __builtin_amdgcn_sched_barrier(0);
                    {
                        const uint8_t *kbn[2], *vbn[2];
                        (void)unit(min(i + 1, gn - 1), kbn, vbn);
                        load_k_half8<kTileBlk>(rk[0], kbn, kRowBytes, koff[0]);
                        load_k_half8<kTileBlk>(rk[1], kbn, kRowBytes, koff[1]);
                        sz = load_scale_zp<kTileBlk>(kbn, vbn, kRowBytes, n16, kg);
                    }
                    pv_half8(st.acc[0], rv[0], pf);
                    pv_half8(st.acc[1], rv[1], pf);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                // r0 holds the first K half of unit i when iteration i begins (loaded by the iteration before; the
                // last iteration loads its own unit's again rather than branching).  No branch in the body: a
                // unit whose blocks are both outside the cache goes through with every score masked.
                HalfRegs r0, r1;
                {
                    const uint8_t *kb[2], *vb[2];
                    (void)unit(0, kb, vb);
                    load_k_half<kTileBlk>(r0, kb, kRowBytes, koff[0]);
                }
                for (int i = 0; i < gn; i++) {
                    const int tok_base = (lb0 + g0 + i) * kUnit;
                    const uint8_t *kb[2], *vb[2];
                    const int ok = unit(i, kb, vb);  // (scalar work: the bases are not carried from iteration to iteration)
                    const bool partial = (tok_base < rg.j0) || (tok_base + kUnit > rg.ctx) || ok != 3;  // wavefront-uniform
                    float4_t sc[2] = {(float4_t){0.f, 0.f, 0.f, 0.f}, (float4_t){0.f, 0.f, 0.f, 0.f}};
                    // (the scheduling barriers keep each half-stage's loads behind the use of the registers
                    // they overwrite: hoisted to the top of the iteration they would all be live at once)
                    load_k_half<kTileBlk>(r1, kb, kRowBytes, koff[1]);
                    scores_half<kBf16>(sc, r0, qf[0]);
                    __builtin_amdgcn_sched_barrier(0);
                    load_v_half<kTileBlk>(r0, vb, kRowBytes, voff[0], v_ok[0]);
                    scores_half<kBf16>(sc, r1, qf[1]);
                    const typename Op16<kBf16>::vec8 pf = softmax_unit<kBf16>(st, sc, c, tok_base, rg.j0, rg.ctx, kg, ok);
                    __builtin_amdgcn_sched_barrier(0);
                    load_v_half<kTileBlk>(r1, vb, kRowBytes, voff[1], v_ok[1]);
                    pv_half<kBf16>(st.acc[0], r0, pf, partial, tok_base, rg.j0, rg.ctx, kg, ok);
                    __builtin_amdgcn_sched_barrier(0);
                    {
                        const uint8_t *kbn[2], *vbn[2];
                        (void)unit(min(i + 1, gn - 1), kbn, vbn);
                        load_k_half<kTileBlk>(r0, kbn, kRowBytes, koff[0]);
                    }
                    pv_half<kBf16>(st.acc[1], r1, pf, partial, tok_base, rg.j0, rg.ctx, kg, ok);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }

        // ---- this wavefront's result for the segment
        float l = st.l, corr = st.corr;
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        if constexpr (kU8) {
            corr += __shfl_xor(corr, 16, 64);
            corr += __shfl_xor(corr, 32, 64);
        }
        const int64_t slot = (int64_t)w + (int64_t)s * Hkv + h;  // unique per (piece, segment)
        if (n16 < G) {
            if (whole && p.sinks != nullptr && l > 0.0f) l += fast_exp2(p.sinks[h * G + n16] * kLog2e - st.m);
            const float inv = whole ? (l > 0.0f ? 1.0f / l : 0.0f) : 1.0f;
#pragma unroll
            for (int half = 0; half < 2; half++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float o[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) o[e] = (kU8 ? st.acc[half][e][r] - corr : st.acc[half][e][r]) * inv;
                    const int d0 = half * 128 + (kg * 4 + r) * 8;
                    if (kPad && d0 >= kHD) continue;  // (columns beyond the head size hold nothing)
                    if (whole) {
                        store_out8(p.out, ((int64_t)rg.token * p.num_heads_q + h * G + n16) * kHD + d0, p.out_dtype, o);
                    } else {
                        float* po = p.part_out + (slot * G + n16) * kHD + d0;
                        *(float4*)(po) = make_float4(o[0], o[1], o[2], o[3]);
                        *(float4*)(po + 4) = make_float4(o[4], o[5], o[6], o[7]);
                    }
                }
            if (!whole && kg == 0) {
                p.part_ml[(slot * G + n16) * 2] = st.m;
                p.part_ml[(slot * G + n16) * 2 + 1] = l;
            }
        }
        L += n;
    }
}

// Combines the partials of every (sequence, kv head) segment that more than one piece worked
// on.  A separate launch: the kernel boundary is what makes the partials visible, which is far
// cheaper here than device-scope fences inside the streaming kernel (those write back and
// invalidate whole L2 caches and cost the decode kernel almost half of its bandwidth).
// kParts == 1: a workgroup per segment, a wavefront per query head of the group (many segments of a few pieces
// each).  Otherwise a workgroup of kParts wavefronts per (segment, query head).
template <int kParts>
__global__ __launch_bounds__(kParts == 1 ? 256 : 64 * kParts) void paged_merge_kernel(PagedParams p) {
    __shared__ float4 shares[kParts == 1 ? 1 : kParts - 1][64];
    const int Hkv = p.num_heads_kv, G = p.num_heads_q / p.num_heads_kv;
    const int seg = kParts == 1 ? blockIdx.x : blockIdx.x / G, s = seg / Hkv, h = seg % Hkv;
    const DecodeRange rg = ((const DecodeRange*)p.seq_info)[s];
    if (rg.nb <= 0) return;
    const int64_t total = (int64_t)p.blk_prefix[p.num_rows] * Hkv;
    if (total <= 0) return;
    const Line line(total, working_waves(p, total, p.overlap ? p.plan_waves[0] : p.num_waves), p.dyn_pieces);
    const int seglen = rg.nb + p.switch_cost;
    const int64_t L0 = (int64_t)p.blk_prefix[s] * Hkv + (int64_t)h * seglen + p.switch_cost, L1 = L0 + rg.nb;
    const int id_first = line.piece_at(L0), id_last = line.piece_at(L1 - 1);
    if (id_first >= id_last) return;  // a single piece covered the segment and wrote the final rows
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if constexpr (kParts == 1) {
        for (int g = wave; g < G; g += 4) merge_segment_head<1>(p, line, s, h, g, rg.token, id_first, id_last, 0, lane, shares);
    } else {
        merge_segment_head<kParts>(p, line, s, h, blockIdx.x % G, rg.token, id_first, id_last, wave, lane, shares);
    }
}

// The most 32-token blocks of a row, and pieces of one segment, that the caller's bound on the contexts allows.
static int64_t most_blocks(const PagedParams& p) {
    int64_t tokens = p.max_context_len > 0 ? p.max_context_len : 0x7fffffff;
    if (p.sliding_window > 0) tokens = std::min(tokens, (int64_t)p.sliding_window + 31);
    return (tokens + 31) / 32;
}
static int64_t most_waves(const PagedParams& p) {
    return working_waves(p, (int64_t)p.num_rows * p.num_heads_kv * (most_blocks(p) + p.switch_cost), p.num_waves);
}

static hipError_t launch_merge(const PagedParams& p, hipStream_t stream) {
    const int segments = p.num_rows * p.num_heads_kv, G = p.num_heads_q / p.num_heads_kv;
    // (few segments of many pieces: 16,384 tokens of one sequence, 64 pieces a segment: the step 23.8 us with four wavefronts
    // to a query head, 23.0 with eight; one wavefront taking piece after piece, as this kernel did: 14.6 us for the merge of 25.
    // Up to eight pieces one wavefront has under way at once: 16 sequences of 100 tokens 13.5 us with eight of them to a head, 12.8 with one)
    if (segments <= 128 && std::min(most_blocks(p), most_waves(p) / segments + 2) > 8)
        hipLaunchKernelGGL(paged_merge_kernel<8>, dim3(segments * G), dim3(512), 0, stream, p);
    else
        hipLaunchKernelGGL(paged_merge_kernel<1>, dim3(segments), dim3(256), 0, stream, p);
    return hipGetLastError();
}

// Schedule options: process-wide, changed with set_option (hipattn_set_option in the C ABI).  The
// environment variable HIPATTN_<NAME IN CAPITALS> gives an option its initial value; the
// environment is read once, when the first option is looked at, never on the call path.
namespace {
struct Option {
    const char* name;
    const char* env;
    int dflt, lo, hi;
    std::atomic<int> value;
};
Option g_options[] = {
    // 0: one kernel after the other for mixed batches; 1: decode beside the chunks' flash kernel
    {"mixed_overlap", "HIPATTN_MIXED_OVERLAP", 1, 0, 1, {1}},
    // block-times a (sequence, kv head) segment start is charged on the decode work line
    {"decode_switch_cost", "HIPATTN_DECODE_SWITCH_COST", 5, 0, 64, {5}},
    // on-demand pieces per wavefront for the last quarter of the decode work line (0: none)
    {"decode_dyn_pieces_per_wave", "HIPATTN_DECODE_DYN_PIECES_PER_WAVE", 0, 0, 64, {0}},
    // scales the compute units the plan gives the decode part of a mixed batch (100 = as modelled)
    {"mixed_decode_share_percent", "HIPATTN_MIXED_DECODE_SHARE_PERCENT", 100, 10, 1000, {100}},
    // 1: dense SDPA at head sizes below 128 runs the tuned head-128 kernel on rows of fewer columns; 0: the plain kernels
    {"sdpa_padded_rows", "HIPATTN_SDPA_PADDED_ROWS", 1, 0, 1, {1}},
    // 1: the decode kernels that have the code for it (u8 caches) combine the partials of split segments
    // themselves; 0: a merge launch behind every decode kernel
    {"decode_fused_merge", "HIPATTN_DECODE_FUSED_MERGE", 1, 0, 1, {1}},
    // dense SDPA in the kernel of sdpa_narrow.hip: 0 never, 1 where it is the faster one, 2 wherever it takes the call
    {"sdpa_narrow", "HIPATTN_SDPA_NARROW", 1, 0, 2, {1}},
    // wavefronts of that kernel that share 32 query rows: 1, 2 or 4; 0: by the time they would take
    {"sdpa_narrow_split", "HIPATTN_SDPA_NARROW_SPLIT", 0, 0, 4, {0}},
};
enum { kOptMixedOverlap = 0, kOptSwitchCost, kOptDynPieces, kOptSharePercent, kOptSdpaPadded, kOptFusedMerge, kOptSdpaNarrow, kOptSdpaNarrowSplit };

void init_options_from_environment() {
    static std::once_flag once;
    std::call_once(once, [] {
        for (Option& o : g_options)
            if (const char* e = getenv(o.env)) o.value.store(std::min(std::max(atoi(e), o.lo), o.hi));
    });
}
int option(int which) {
    init_options_from_environment();
    return g_options[which].value.load(std::memory_order_relaxed);
}
}  // namespace

bool sdpa_padded_rows_enabled() { return option(kOptSdpaPadded) != 0; }
int sdpa_narrow_option() { return option(kOptSdpaNarrow); }
int sdpa_narrow_split_option() { return option(kOptSdpaNarrowSplit); }

bool set_option(const char* name, int value) {
    init_options_from_environment();
    for (Option& o : g_options)
        if (strcmp(o.name, name) == 0) {
            o.value.store(value < 0 ? o.dflt : std::min(std::max(value, o.lo), o.hi));
            return true;
        }
    return false;
}

// ---- host side of the fast path ---------------------------------------------------------

// Every head size up to 256 that is a multiple of 8 with 16-bit and u8 caches, on blocks of 16, 32 or a
// larger power of two.

// fp16 queries on a bf16 cache at head size 128: the ordinary launch with the blocks converted to fp16 operands
// (kHalfFromBf16; no self-planning or eight-wavefront form of it is built, nor one with the distance bias).
static bool half_operands_from_bf16(const PagedParams& p) {
    return p.cache_dtype == HIPATTN_BF16 && p.q_dtype == HIPATTN_F16 && p.head_dim == kD && !p.alibi_slopes;
}

bool paged_fast_supported(const PagedParams& p) {
    const int G = p.num_heads_q / p.num_heads_kv;
    if (G > 16 || !(p.q_dtype == HIPATTN_F16 || p.q_dtype == HIPATTN_BF16)) return false;
    // (head sizes below 64 / between 64 and 128: the head-64 / head-128 kernel with zero columns)
    if (p.block_size < 16 || (p.block_size & (p.block_size - 1)) != 0) return false;  // 16, 32, or a larger power of two
    if (p.alibi_slopes && p.head_dim > 128) return false;  // (the head-256 decode kernel has no distance term: the query-tile kernel takes the batch)
    // (above 128: paged_decode256_kernel)
    return p.head_dim >= 8 && p.head_dim <= 256 && p.head_dim % 8 == 0 &&
           (p.cache_dtype == HIPATTN_F16 || p.cache_dtype == HIPATTN_BF16 || p.cache_dtype == HIPATTN_U8);
}

PagedParams split_kv_heads(const PagedParams& p) {
    const int G = p.num_heads_q / p.num_heads_kv;
    if (G <= 16 || p.kv_share != 1) return p;
    for (int share = 2; share <= G; share++) {
        if (G % share != 0 || G / share > 16) continue;
        if (G / share < 8) break;  // (groups that fill less than half of a 16-row product: the K/V rows would be read too often)
        if ((int64_t)p.num_heads_kv * share > 0x7fff) break;
        PagedParams s = p;
        s.num_heads_kv = p.num_heads_kv * share;
        s.kv_share = share;
        return paged_fast_supported(s) ? s : p;
    }
    return p;  // (a prime number of heads, say: the query-tile kernel keeps the call)
}

// The chunk kernels address K and V by the cache's own kv heads.
static PagedParams with_cache_heads(const PagedParams& p) {
    PagedParams r = p;
    r.num_heads_kv = p.num_heads_kv / p.kv_share;
    r.kv_share = 1;
    return r;
}

// Wavefronts the decode kernel keeps resident: it needs up to 256 registers per lane, i.e. two
// wavefronts per SIMD, eight per compute unit.
static int resident_decode_waves() {
    static thread_local int cached_device = -1, cached_waves = 0;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 2048;
    if (dev != cached_device) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
        cached_device = dev;
        cached_waves = cus * 8;
    }
    return cached_waves;
}

// fp16 caches stream best with one wavefront per SIMD (four per compute unit; three measure the
// same); the u8 path has more arithmetic per byte and wants more: six per compute unit measured
// 1.5 % faster than all eight on the 128-sequence u8 configuration, counts that do not divide
// evenly over the compute units 5-10 % slower.
// Upper bound of the 128-row query tiles of the batch's multi-token sequences (the lengths stay
// on the device): each such sequence has at least 2 tokens and wastes at most one tile.
// 0 selects the row-per-token form of the plan, which takes the batch to hold as many rows as
// sequences: only a batch with exactly that many tokens may get it (a single token spread over two
// or more sequences, all but one of them empty, has a bound of 0 by the formula and must not); and one
// token in one sequence, which has no other length.
static int query_tile_bound(const PagedParams& p) {
    if (p.num_tokens == p.num_seqs && (!p.any_lengths || p.num_seqs == 1)) return 0;  // one token per sequence: a pure decode batch
    return std::max(1, p.num_tokens / 128 + std::min(p.num_seqs, p.num_tokens / 2));
}

// Mixed batches run the decode kernel beside the chunks' flash kernel unless the caller fixed the
// number of decode wavefronts or the option mixed_overlap = 0 asks for one kernel after the other.
// Records of the decode plan: one per sequence, or one per token when the batch is planned per token.
static int plan_rows(const PagedParams& p) { return query_tile_bound(p) == 0 ? p.num_tokens : p.num_seqs; }

static bool overlap_wanted(const PagedParams& p) {
    if (query_tile_bound(p) == 0 || p.num_waves > 0 || p.no_side_stream || p.alibi_slopes || half_operands_from_bf16(p)) return false;
    // the eight-wavefront decode kernel: head size 128, and 16-bit caches at the head sizes between 64 and 128
    if (p.head_dim != kD && !(p.head_dim > 64 && p.head_dim < kD && p.cache_dtype != HIPATTN_U8)) return false;
    return option(kOptMixedOverlap) != 0;
}

static int choose_num_waves(const PagedParams& p, bool overlap) {
    if (p.num_waves > 0) return p.num_waves;
    const int resident = resident_decode_waves();
    if (overlap) return resident;  // the most the plan may choose
    // (u8 at head size 64 has the most arithmetic per byte of all: every resident wavefront, 0.59 against
    // 0.48 of HBM peak with six per compute unit on the 128-sequence u8 batch)
    if (p.head_dim > 128) return resident;  // half as many bytes in flight per wavefront: twice the wavefronts
    if (p.cache_dtype == HIPATTN_U8) return p.head_dim <= 64 ? resident : resident / 4 * 3;
    return resident / 2;
}

static size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// On-demand pieces per wavefront for the last quarter of the line.  Off by default: a wavefront
// that starts on a new piece pays a chain of dependent loads (ticket, sequence, block table,
// first block) before it streams again, and on MI355X that costs more than the better balance
// at the end of the kernel wins back.  The option decode_dyn_pieces_per_wave switches it on.
static int choose_dyn_pieces(const PagedParams& p, int num_waves, bool overlap) {
    if (overlap || p.head_dim > 128) return 0;  // (the head-256 kernel has static pieces only)
    return num_waves * option(kOptDynPieces);
}

// Bytes of one slot of unnormalised partial outputs: [G, head_dim] floats for the merge kernel, or the
// fused merge's lane layout (kPartPairs pairs for each of 4 G lanes), whichever is larger.
static size_t part_floats_per_slot(const PagedParams& p) {
    const size_t G = (size_t)(p.num_heads_q / p.num_heads_kv);
    return std::max(G * p.head_dim, (size_t)kPartPairs * 4 * G * 2) * sizeof(float);
}

size_t paged_fast_workspace_bytes(const PagedParams& p) {
    const bool overlap = overlap_wanted(p);
    const int W = choose_num_waves(p, overlap);
    const int G = p.num_heads_q / p.num_heads_kv;
    const size_t rows = (size_t)plan_rows(p);
    const size_t slots = (size_t)W + choose_dyn_pieces(p, W, overlap) + rows * p.num_heads_kv;
    return 512 + 2 * align_up((rows + 1) * sizeof(int32_t), 256) + align_up(rows * 32, 256) +
           align_up(slots * part_floats_per_slot(p), 256) + align_up(slots * G * 2 * sizeof(float), 256) +
           align_up(slots * sizeof(uint64_t), 256);
}

// The chunks of a u8 batch read rows that the prologue has just quantised, 128 query rows at a time, and dequantise them through
// registers in the phase that bounds the chunk kernel.  The rows of sequences without cached tokens are therefore kept in fp16 as
// well, the values that dequantisation gives, at 5 us more for the prologue of 9,000 tokens.  Measured (us a step, 32 heads on 8, without -> with):
// six prompts of 100 to 3,000 tokens 166 -> 149, two of 3,000 205 -> 181, one of 1,000 46 -> 40, eight of 512 beside 120 decode rows (64
// heads) 283 -> 274.  Up to 256 MiB (65,536 tokens of 8 heads).
static int64_t shadow_blocks(const PagedParams& p) { return (int64_t)(p.num_tokens / p.block_size) + p.num_seqs + 1; }

size_t paged_shadow_bytes(const PagedParams& p) {
    if (p.cache_dtype != HIPATTN_U8 || p.head_dim != 128 || !overlap_wanted(p) || !paged_mixed_supported(p)) return 0;
    if (p.num_tokens < kShadowTokens || (p.max_context_len > 0 && p.max_context_len < kShadowTokens)) return 0;
    const int64_t kv_heads = p.num_heads_kv / p.kv_share;
    const size_t rows = (size_t)(shadow_blocks(p) * kv_heads * p.block_size) * 128 * sizeof(uint16_t);
    return rows > (size_t)128 << 20 ? 0 : 256 + 2 * rows + align_up((size_t)shadow_blocks(p) * sizeof(int32_t), 256);
}

// A value no earlier call of this process used and that memory which was never written is unlikely to hold.
static unsigned long long next_merge_tag() {
    static std::atomic<unsigned long long> counter{0};
    static const unsigned long long base = [] {
        unsigned long long x = 0x9e3779b97f4a7c15ull ^ (unsigned long long)(uintptr_t)&counter;
        x ^= (unsigned long long)std::chrono::steady_clock::now().time_since_epoch().count() * 0xbf58476d1ce4e5b9ull;
        return x | (1ull << 63);
    }();
    return base + (counter.fetch_add(1, std::memory_order_relaxed) << 1) + 1;  // never zero: zero means "taken"
}


void paged_fast_plan(PagedParams& p, void* workspace, size_t workspace_bytes) {
    const bool overlap = overlap_wanted(p);  // asks whether the caller fixed num_waves: before it is filled in
    const size_t shadow = p.no_side_stream ? 0 : paged_shadow_bytes(p);
    p.overlap = overlap ? 1 : 0;
    const bool fixed_waves = p.num_waves > 0;
    p.num_waves = choose_num_waves(p, overlap);
    p.switch_cost = option(kOptSwitchCost);
    p.dyn_pieces = choose_dyn_pieces(p, p.num_waves, overlap);
    p.overlap_share = option(kOptSharePercent) / 100.0f;
    p.dyn_groups = std::min(64, std::max(1, p.num_waves / 32));  // every group has at least one wavefront
    const int G = p.num_heads_q / p.num_heads_kv;
    p.max_q_tiles = query_tile_bound(p);
    p.num_rows = plan_rows(p);
    // One sequence: its length is known to the device alone, and it may turn out to be a single token (a padded or a recorded call).  As a
    // decode row that needs the decode workgroups and the merge, which cost every prompt 2 us (64 tokens 14.5 -> 16.5, 1,000 38.0 -> 40.1); as
    // a query tile it needs neither, but walks its context alone (us, tile / decode row: 300 tokens 21 / 16, 2,000 54 / 19, 8,000 165 / 23; u8
    // 22 / 18, 70 / 21, 236 / 23).  A tile while the bound on the context keeps it below 45 us, which two kernels took for any context.
    p.lone_tile = overlap && p.num_seqs == 1 && most_blocks(p) <= 32 && paged_mixed_supported(p) ? 1 : 0;
    const int64_t segments = (int64_t)p.num_rows * p.num_heads_kv;
    // 16-bit caches: from 128 segments on all wavefronts (24 sequences of 400: 16.1 us against 17.4 with 512; 63 of 300, 504
    // segments: 23.1 against 23.8 with 768).  (On-demand pieces: every ticket group needs its wavefronts.)
    const bool all = fixed_waves || option(kOptDynPieces) > 0 || overlap || (p.cache_dtype != HIPATTN_U8 && segments >= 128);
    p.few_waves = all ? 0 : (int)std::max<int64_t>(512, 2 * segments);
    const size_t slots = (size_t)p.num_waves + p.dyn_pieces + (size_t)p.num_rows * p.num_heads_kv;
    uint8_t* w = (uint8_t*)workspace;
    p.dyn_counter = (int32_t*)w;
    w += 256;
    p.plan_waves = (int32_t*)w;
    w += 256;
    p.tile_prefix = (int32_t*)w;
    w += align_up(((size_t)p.num_rows + 1) * sizeof(int32_t), 256);
    p.blk_prefix = (int32_t*)w;
    w += align_up(((size_t)p.num_rows + 1) * sizeof(int32_t), 256);
    p.seq_info = w;
    w += align_up((size_t)p.num_rows * 32, 256);
    p.part_out = (float*)w;
    w += align_up(slots * part_floats_per_slot(p), 256);
    p.part_ml = (float*)w;
    w += align_up(slots * G * 2 * sizeof(float), 256);
    p.part_flag = (uint64_t*)w;
    w += align_up(slots * sizeof(uint64_t), 256);
    if (shadow > 0 && (size_t)(w - (uint8_t*)workspace) + shadow <= workspace_bytes) {
        w += (256 - (uintptr_t)w % 256) % 256;
        const size_t rows = (size_t)(shadow_blocks(p) * (p.num_heads_kv / p.kv_share) * p.block_size) * 128;
        p.shadow_k = (uint16_t*)w;
        p.shadow_v = p.shadow_k + rows;
        p.shadow_table = (int32_t*)(p.shadow_v + rows);
    }
    // the head-256 kernel and on-demand pieces (whose order of completion is not that of their numbers) keep the merge launch
    // Built into the u8 kernels only (see kFusedBuilt).  Measured, whole steps on one machine: the 128-sequence
    // u8 batch 0.437 ms fused against 0.440 ms with the merge launch.  Where many pieces share a segment the one wavefront that
    // combines them in the kernel takes them two by two: one sequence of 778 tokens 36 against 12.5 us, of 16,384 88 against 24,
    // 32 sequences of 4,000 (256 segments) 75 against 69, 64 of them (512 segments) 127 against 127: fused up to three pieces to a
    // segment (49 sequences of 300: 20.4 against 22.4), two and a half at head size 64 (172 segments of 283: 21.0 against 19.3 with
    // three), and up to two blocks, of which each may be a piece, or four in many segments (40 of 100: 15.0 against 17.6; 16 heads' 32
    // segments of 81: 13.3 against 12.6).  Beside a chunk kernel the launch costs the host 8 us: up to eight blocks (a prompt of
    // 60 tokens 35.5 against 44.5).
    const bool few_pieces = fixed_waves || most_blocks(p) <= (overlap ? 8 : segments >= 128 ? 4 : 2) ||
                            2 * most_waves(p) <= (p.head_dim <= 64 ? 5 : 6) * segments;
    p.fused_merge = (option(kOptFusedMerge) != 0 && p.cache_dtype == HIPATTN_U8 && p.dyn_pieces == 0 && p.head_dim <= 128 && few_pieces) ? 1 : 0;
    p.merge_tag = next_merge_tag();
}

// ---- scratch of the entry point that allocates nothing (hipattn_paged_attention_noalloc) ------
// A file-scope device array stands in for the caller's workspace: every GPU the library runs on
// holds its own copy until the process ends.  In host code the array's name is not a device
// address; the address on the current device comes from hipGetSymbolAddress, once per device, and
// that pointer is what kernels and host calls get.  Calls that overlap on one GPU share the array
// and race; it keeps the previous call's contents (the plan clears the ticket counters, everything
// else is written before it is read).
constexpr size_t kStaticScratchBytes = HIPATTN_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) uint8_t scratch[kStaticScratchBytes];

hipError_t paged_static_scratch(void** ptr, size_t* bytes) {
    static std::mutex mutex;
    static void* address[64] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> guard(mutex);
    if (!address[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        address[dev] = p;
    }
    *ptr = address[dev];
    *bytes = kStaticScratchBytes;
    return hipSuccess;
}

// A side stream and a fork/join pair of events per (device, caller's stream), made on the first
// mixed batch that stream carries, so that mixed batches on different streams do not wait for each
// other's chunk kernels.  An entry lives until its stream is destroyed through the C ABI
// (release_side_stream) or the process ends; beyond kMaxSideStreams entries further caller streams
// share the device's first entry.  The entry's mutex keeps the record/wait pairs of concurrent
// callers apart.
struct SideStream {
    int device = 0;
    hipStream_t owner = nullptr;
    hipStream_t stream = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
    std::mutex mutex;
};

constexpr int kMaxSideStreams = 32;
static std::mutex g_side_mutex;
static SideStream* g_side[kMaxSideStreams] = {};

static SideStream* side_stream(hipStream_t owner) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> guard(g_side_mutex);
    int free_slot = -1;
    SideStream* shared = nullptr;
    for (int i = 0; i < kMaxSideStreams; i++) {
        SideStream* s = g_side[i];
        if (!s) {
            if (free_slot < 0) free_slot = i;
            continue;
        }
        if (s->device != dev) continue;
        if (s->owner == owner) return s;
        if (!shared) shared = s;
    }
    if (free_slot < 0) return shared;  // table full: share (nullptr if this device has none, the caller reports it)
    SideStream* s = new SideStream;
    s->device = dev;
    s->owner = owner;
    if (hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&s->fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&s->join, hipEventDisableTiming) != hipSuccess) {
        if (s->stream) (void)hipStreamDestroy(s->stream);
        if (s->fork) (void)hipEventDestroy(s->fork);
        if (s->join) (void)hipEventDestroy(s->join);
        delete s;
        return nullptr;
    }
    g_side[free_slot] = s;
    return s;
}

// Called before a stream is destroyed: whatever its side stream still runs is waited for, then the
// side stream and its events go.  Streams other callers share through a full table are not owned by
// the stream being destroyed and stay.
void release_side_stream(hipStream_t owner) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return;
    SideStream* s = nullptr;
    {
        std::lock_guard<std::mutex> guard(g_side_mutex);
        for (int i = 0; i < kMaxSideStreams; i++)
            if (g_side[i] && g_side[i]->device == dev && g_side[i]->owner == owner) {
                s = g_side[i];
                g_side[i] = nullptr;
                break;
            }
    }
    if (!s) return;
    {
        std::lock_guard<std::mutex> guard(s->mutex);
        (void)hipStreamSynchronize(s->stream);
        (void)hipStreamDestroy(s->stream);
        (void)hipEventDestroy(s->fork);
        (void)hipEventDestroy(s->join);
    }
    delete s;
}

// The decode kernel for p's cache type, head size and block size (a combination paged_fast_supported
// admits; head sizes other than 128 have the ordinary form only, blocks of more than 32 tokens no self-planning form).
template <bool kU8, bool kBf16, int kWaves, bool kSelfPlan, int kHD, bool kPad>
static void launch_decode_blk(const PagedParams& p, const KvWriteParams& wp, int do_write, dim3 grid, dim3 block, hipStream_t stream) {
    if constexpr (kWaves == 1 && !kSelfPlan && kBf16 && kHD == 128 && !kPad) {
        if (half_operands_from_bf16(p)) {
            if (p.block_size == 32)
                hipLaunchKernelGGL((paged_decode_kernel<false, false, 1, false, 128, 32, false, false, true>), grid, block, 0, stream, p, wp, do_write);
            else if (p.block_size == 16)
                hipLaunchKernelGGL((paged_decode_kernel<false, false, 1, false, 128, 16, false, false, true>), grid, block, 0, stream, p, wp, do_write);
            else
                hipLaunchKernelGGL((paged_decode_kernel<false, false, 1, false, 128, 0, false, false, true>), grid, block, 0, stream, p, wp, do_write);
            return;
        }
    }
    if constexpr (kWaves == 1 && !kSelfPlan) {
        if (p.alibi_slopes) {  // the instantiations with the distance bias
            if (p.block_size == 32)
                hipLaunchKernelGGL((paged_decode_kernel<kU8, kBf16, 1, false, kHD, 32, kPad, true>), grid, block, 0, stream, p, wp, do_write);
            else if (p.block_size == 16)
                hipLaunchKernelGGL((paged_decode_kernel<kU8, kBf16, 1, false, kHD, 16, kPad, true>), grid, block, 0, stream, p, wp, do_write);
            else
                hipLaunchKernelGGL((paged_decode_kernel<kU8, kBf16, 1, false, kHD, 0, kPad, true>), grid, block, 0, stream, p, wp, do_write);
            return;
        }
    }
    if (p.block_size == 32) {
        hipLaunchKernelGGL((paged_decode_kernel<kU8, kBf16, kWaves, kSelfPlan, kHD, 32, kPad>), grid, block, 0, stream, p, wp, do_write);
    } else if (p.block_size == 16) {
        hipLaunchKernelGGL((paged_decode_kernel<kU8, kBf16, kWaves, kSelfPlan, kHD, 16, kPad>), grid, block, 0, stream, p, wp, do_write);
    } else if constexpr (!kSelfPlan) {
        hipLaunchKernelGGL((paged_decode_kernel<kU8, kBf16, kWaves, false, kHD, 0, kPad>), grid, block, 0, stream, p, wp, do_write);
    }
}

template <bool kBf16, bool kPad, bool kU8 = false>
static void launch_decode256_blk(const PagedParams& p, dim3 grid, dim3 block, hipStream_t stream) {
    if (p.block_size == 32)
        hipLaunchKernelGGL((paged_decode256_kernel<kBf16, 32, kPad, kU8>), grid, block, 0, stream, p);
    else if (p.block_size == 16)
        hipLaunchKernelGGL((paged_decode256_kernel<kBf16, 16, kPad, kU8>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((paged_decode256_kernel<kBf16, 0, kPad, kU8>), grid, block, 0, stream, p);
}

template <int kWaves, bool kSelfPlan>
static void launch_decode(const PagedParams& p, const KvWriteParams& wp, int do_write, dim3 grid, dim3 block,
                          hipStream_t stream) {
    const bool bf16 = p.cache_dtype == HIPATTN_BF16, u8 = p.cache_dtype == HIPATTN_U8;
    if (p.head_dim == 128) {
        if (u8)
            launch_decode_blk<true, false, kWaves, kSelfPlan, 128, false>(p, wp, do_write, grid, block, stream);
        else if (bf16)
            launch_decode_blk<false, true, kWaves, kSelfPlan, 128, false>(p, wp, do_write, grid, block, stream);
        else
            launch_decode_blk<false, false, kWaves, kSelfPlan, 128, false>(p, wp, do_write, grid, block, stream);
    } else if constexpr (kWaves == 8) {  // (overlap_wanted: 16-bit caches at head sizes between 64 and 128)
        if (bf16)
            launch_decode_blk<false, true, 8, false, 128, true>(p, wp, do_write, grid, block, stream);
        else
            launch_decode_blk<false, false, 8, false, 128, true>(p, wp, do_write, grid, block, stream);
    } else if constexpr (kWaves == 1 && !kSelfPlan) {
        if (p.head_dim > 128) {
            if (p.head_dim == 256) {
                if (u8) launch_decode256_blk<false, false, true>(p, grid, block, stream);
                else if (bf16) launch_decode256_blk<true, false>(p, grid, block, stream);
                else launch_decode256_blk<false, false>(p, grid, block, stream);
            } else {
                if (u8) launch_decode256_blk<false, true, true>(p, grid, block, stream);
                else if (bf16) launch_decode256_blk<true, true>(p, grid, block, stream);
                else launch_decode256_blk<false, true>(p, grid, block, stream);
            }
        } else if (p.head_dim == 64) {
            if (u8) launch_decode_blk<true, false, 1, false, 64, false>(p, wp, do_write, grid, block, stream);
            else if (bf16) launch_decode_blk<false, true, 1, false, 64, false>(p, wp, do_write, grid, block, stream);
            else launch_decode_blk<false, false, 1, false, 64, false>(p, wp, do_write, grid, block, stream);
        } else if (p.head_dim > 64) {
            if (u8) launch_decode_blk<true, false, 1, false, 128, true>(p, wp, do_write, grid, block, stream);
            else if (bf16) launch_decode_blk<false, true, 1, false, 128, true>(p, wp, do_write, grid, block, stream);
            else launch_decode_blk<false, false, 1, false, 128, true>(p, wp, do_write, grid, block, stream);
        } else {
            if (u8) launch_decode_blk<true, false, 1, false, 64, true>(p, wp, do_write, grid, block, stream);
            else if (bf16) launch_decode_blk<false, true, 1, false, 64, true>(p, wp, do_write, grid, block, stream);
            else launch_decode_blk<false, false, 1, false, 64, true>(p, wp, do_write, grid, block, stream);
        }
    }
}

hipError_t launch_paged_fast(const PagedParams& params, const KvWriteParams* write, hipStream_t stream,
                             const KernelProbe& probe) {
    PagedParams p = params;
    KvWriteParams wp{};
    int write_blocks = 0;
    if (write) {
        wp = *write;
        if (wp.head_dim > 256) return hipErrorInvalidValue;  // the fast path is head sizes up to 256 only
        write_blocks = (int)((kv_write_wavefronts(wp) + 3) / 4);
    }
    if (wp.vector_rows)
        wp.shadow_k = p.shadow_k, wp.shadow_v = p.shadow_v, wp.shadow_table = p.shadow_table;
    else
        p.shadow_table = nullptr;  // (nobody to fill it)
    hipError_t e = hipSuccess;
    // A pure decode batch of few rows is one launch less: the decode wavefronts plan for themselves
    // and write the new rows (see kSelfPlanMaxRows).
    const bool self_plan = p.max_q_tiles == 0 && p.num_rows <= kSelfPlanMaxRows && p.dyn_pieces == 0 && p.head_dim == kD &&
                           p.block_size <= 32 && (!write || wp.vector_rows) && !p.alibi_slopes && !half_operands_from_bf16(p);
    if (self_plan) {
        if (probe.before) (void)hipEventRecord(probe.before, stream);
        launch_decode<1, true>(p, wp, write ? 1 : 0, dim3(p.num_waves), dim3(64), stream);
        e = hipGetLastError();
        if (probe.after) (void)hipEventRecord(probe.after, stream);
        if (e != hipSuccess || p.fused_merge) return e;
        return launch_merge(p, stream);
    }
    // prologue: KV-cache write of the new tokens (optional) + plan, one launch
    hipLaunchKernelGGL(paged_prologue_kernel, dim3(write_blocks + 1), dim3(256), 0, stream, wp, p, write_blocks);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    // Shapes without the eight-wavefront decode kernel run the two parts side by side all the same when
    // the decode wavefronts take at most half of every compute unit's registers (and no LDS), so that the
    // chunks' workgroups find room beside them.
    const bool beside = p.max_q_tiles > 0 && !p.overlap && !p.no_side_stream && !p.alibi_slopes && option(kOptMixedOverlap) != 0 &&
                        p.num_waves * 2 <= resident_decode_waves();
    if (p.overlap && paged_mixed_supported(p)) {
        if (probe.before) (void)hipEventRecord(probe.before, stream);
        e = launch_paged_mixed(p, p.num_heads_kv / p.kv_share, stream);
        if (probe.after) (void)hipEventRecord(probe.after, stream);
        return e != hipSuccess || p.fused_merge || p.lone_tile ? e : launch_merge(p, stream);
    }
    if (p.max_q_tiles > 0 && (p.overlap || beside)) {
        // Mixed batch of a shape that the kernel of both parts (paged_mixed.hip) does not take: the decode
        // sequences stream from HBM on a few compute units while the
        // chunks' flash kernel, on a side stream, has the others; both only need the prologue's
        // results.  The decode kernel stays on the caller's stream, directly behind the prologue,
        // so that it is dispatched first and gets its compute units at once.
        SideStream* side = side_stream(stream);
        if (!side) return hipErrorOutOfMemory;
        std::lock_guard<std::mutex> guard(side->mutex);
        if ((e = hipEventRecord(side->fork, stream)) != hipSuccess) return e;
        if ((e = hipStreamWaitEvent(side->stream, side->fork, 0)) != hipSuccess) return e;
        if (probe.before) (void)hipEventRecord(probe.before, stream);
        if (p.overlap)
            launch_decode<8, false>(p, wp, 0, dim3(p.num_waves / 8), dim3(512), stream);
        else
            launch_decode<1, false>(p, wp, 0, dim3(p.num_waves), dim3(64), stream);
        e = hipGetLastError();
        if (probe.after) (void)hipEventRecord(probe.after, stream);
        const hipError_t e_prefill = launch_paged_prefill(with_cache_heads(p), side->stream);
        if (e == hipSuccess && !p.fused_merge) e = launch_merge(p, stream);
        // always join, also after an error, so the caller's stream never runs ahead of the side stream
        hipError_t e_join = hipEventRecord(side->join, side->stream);
        if (e_join == hipSuccess) e_join = hipStreamWaitEvent(stream, side->join, 0);
        return e != hipSuccess ? e : (e_prefill != hipSuccess ? e_prefill : e_join);
    }
    if (probe.before) (void)hipEventRecord(probe.before, stream);
    launch_decode<1, false>(p, wp, 0, dim3(p.num_waves), dim3(64), stream);
    e = hipGetLastError();
    if (probe.after) (void)hipEventRecord(probe.after, stream);
    if (e != hipSuccess) return e;
    if (!p.fused_merge) {
        e = launch_merge(p, stream);
        if (e != hipSuccess) return e;
    }
    if (p.max_q_tiles > 0) {
        e = launch_paged_prefill(with_cache_heads(p), stream);
    }
    return e;
}

}  // namespace hipattn
