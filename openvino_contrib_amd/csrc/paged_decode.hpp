// Paged-attention decode for gfx950 (sequences with exactly one new token), scheduled
// stream-K style over the whole batch.
//
// Work decomposition.  The unit of work is 32 tokens of the cache of one kv head of one sequence
// -- one cache block of 32 tokens, two of 16, or a 32-token part of a larger one ("block-head": at head size 128, 8 KiB of K plus
// 8 KiB of V in fp16, 2 x 4352 B in u8).  All
// block-heads of the batch are laid out on one line, ordered (sequence, kv head, block), and
// the line is cut into `num_waves` equal pieces; wavefront w owns piece w.  The kernel is
// launched with exactly as many single-wavefront workgroups as fit on the device at once, so
// every wavefront streams the same number of bytes and they all finish together: no tail, no
// per-chunk launch cost, no dependence on how the contexts happen to be distributed.  A piece
// that covers a whole (sequence, kv head) segment writes the final output rows; otherwise the
// wavefront leaves a partial (running max, sum, unnormalised output) per query head in the
// workspace and paged_merge_kernel combines the pieces of a segment with a log-sum-exp
// reduction.  The
// per-sequence block counts and their prefix sum come from the plan workgroup of the prologue
// kernel, which reads past_lens / subsequence_begins on the device: the host never sees the
// lengths.  The same launch performs the operator's KV-cache write.
//
// One wavefront serves the whole GQA group (all query heads sharing the kv head, up to 16),
// so every KV byte is read from HBM exactly once.  Per block it streams K and V straight from
// global memory into MFMA operand registers (two register stages: the next block's loads are
// in flight while the current block is consumed) and keeps an online softmax.
//
// MFMA use (v_mfma_f32_16x16x32_f16; _bf16 for bf16 caches).  Scores are computed transposed, S^T = K Q^T, with the
// 16 tokens of a tile on the M side and the (padded) 16 query heads on the N side; the
// accumulator layout then gives each lane four consecutive tokens of one head, which is
// exactly the B-operand layout the second product O^T = V^T P^T needs, so P never moves
// between lanes.  The contraction index of an MFMA can be permuted freely as long as both
// operands use the same permutation; that freedom is used to make every global load a
// contiguous 16-byte (fp16, bf16) or 8-byte (u8) piece of a cache row:
//   K operand: lane (tok = lane & 15, kg = lane >> 4) holds K[tok][kg*32 + i*8 .. +8], i = 0..3
//   V operand: lane (c = lane & 15, kg) loads V[tok(kg,j)][c*8 .. +8] for its 8 tokens j and
//              transposes the 8x8 patch in registers; MFMA e then yields O[:, c*8 + e].
// u8 caches are dequantised in registers: bytes become exact fp16 integers, the per-token
// scale is folded into the score / probability and the zero-point into a rank-one
// correction (q.(k - zp) s = s (q.k) - s zp sum(q)).
//
// Shapes.  The kernel is a template over the head size it is built for (128 or 64: a lane's K
// piece count and the number of MFMAs per tile follow), the cache block size (32, 16, or 0: a larger power of two read from the call) and whether
// the call's head size may be smaller than the built one (any multiple of 8: rows are then
// head_dim elements apart at run time and the query columns that do not exist are zeros).  The
// figures and layouts above are those of head size 128.
//
// Mixed batches (decode sequences and multi-token chunks in one call).  The chunks are worked on by the flash
// loop over the block table, which is bound by the matrix cores; the decode sequences are bound
// by HBM.  Each of the two needs whole compute units (registers, LDS), so they cannot
// share one, but they can share the chip: paged_mixed.hip runs both in one launch, the decode part with eight
// wavefronts to a workgroup -- a workgroup owns a compute unit -- in the workgroups dispatched first, the chunks
// in those behind them, on the other compute units (and every one the decode workgroups give back).  How many compute units the
// decode part keeps is decided by the plan on the device, in proportion to the work of the two
// parts (cache bytes to stream against key tiles to multiply), so that both end together;
// workgroups beyond that number leave at once.
//
// No counterpart in the reference: its decode path copies the whole contiguous KV state
// three times per token (src/cuda_variable_state.hpp:135-160, src/ops/read_value.cpp:65-71,
// src/ops/assign.cpp:52-54) and materialises the scores in HBM (src/ops/matmul.cpp:204-226,
// src/ops/softmax.cpp:184-192).
#pragma once

#include <type_traits>

#include "decode_operands.hpp"
#include "device_common.hpp"
#include "kernels.hpp"
#include "kv_cache_write.hpp"

namespace hipattn {

constexpr int kD = 128;   // head size of the benchmark configurations (the kernels also take 64 and, padded, any multiple of 8 below: templates kHD, kPad)
constexpr int kBS = 32;   // their cache block size (also 16: template kBlk)
constexpr int kUnit = 32; // tokens a wavefront works through at a time: one block of 32, or two of 16

struct alignas(32) DecodeRange {
    int write_pos;    // cache position of the row's own new token when it has a slot in the table, else -1
    int token;        // row of q / out
    int ctx;          // attended positions end (exclusive)
    int j0;           // attended positions begin
    int new_begin;    // cache position of the first token its sequence contributes to this batch (past_lens)
    int nb;           // number of 32-token units attended (0 when not valid)
    int table_begin;  // offset of the sequence's block table in block_indices
    int empty_row;    // a single-token row with nothing to attend: its output row is zeros
};
static_assert(sizeof(DecodeRange) == 32, "one 32-byte record per sequence");

// Sequence that owns token t: the last s with subsequence_begins[s] <= t.
__device__ __forceinline__ int sequence_of_token(const PagedParams& p, int t) {
    int lo = 0, hi = p.num_seqs;  // begins[lo] <= t < begins[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (p.subsequence_begins[mid] <= t)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// Range of cache positions a single-token row attends.  Computed once per call by the plan and
// stored per record (seq_info), so that the decode and merge kernels fetch it with one load.
//
// Records are per sequence when the batch may hold multi-token sequences (max_q_tiles > 0: those go
// to the chunked-prefill kernel and only sequences of exactly one token are decode rows).  A batch
// with as many tokens as sequences is planned per TOKEN instead (max_q_tiles == 0, no prefill
// launch): record i is token i, whichever sequence it belongs to, so a batch that only looks like
// a decode step -- an empty sequence beside a two-token one -- still gets every row right; its
// extra tokens are simply decode rows with their own context length.
__device__ __forceinline__ DecodeRange decode_range(const PagedParams& p, int i) {
    DecodeRange r;
    int s = i, pos_in_seq = 0;
    bool single = true;
    // everything a row of an ordinary decode batch needs is fetched at once, on the guess that row i is
    // sequence i (one level of memory latency instead of two); a guess that fails is redone below
    // (rows beyond the last sequence exist only when rows are tokens: the guess is then made on the last sequence)
    const int ig = min(i, p.num_seqs - 1);
    const int b0 = p.subsequence_begins[ig], b1 = p.subsequence_begins[ig + 1];
    int tb0 = p.block_indices_begins[ig], tb1 = p.block_indices_begins[ig + 1], past = p.past_lens[ig];
    if (p.max_q_tiles == 0) {
        if (!(ig == i && b0 == i && b1 == i + 1)) {
            s = sequence_of_token(p, i);
            tb0 = p.block_indices_begins[s];
            tb1 = p.block_indices_begins[s + 1];
            past = p.past_lens[s];
        }
        pos_in_seq = i - p.subsequence_begins[s];
        r.token = i;
        // a token outside every sequence (padding in front of the first or behind the last): no row at all
        single = i >= p.subsequence_begins[0] && i < p.subsequence_begins[p.num_seqs];
    } else {
        r.token = b0;
        single = (b1 - b0 == 1);
    }
    const int table_tokens = (tb1 - tb0) * p.block_size;
    r.ctx = min(past + pos_in_seq + 1, table_tokens);
    r.j0 = 0;
    if (p.sliding_window > 0 && r.ctx - p.sliding_window > 0) r.j0 = r.ctx - p.sliding_window;
    const bool valid = single && r.ctx > 0;
    r.write_pos = (single && past + pos_in_seq < table_tokens) ? past + pos_in_seq : -1;
    r.empty_row = single && r.ctx <= 0;
    r.new_begin = past;
    r.nb = valid ? (r.ctx + kUnit - 1) / kUnit - r.j0 / kUnit : 0;  // in units of 32 tokens
    r.table_begin = tb0;
    return r;
}

#ifndef HIPATTN_U8_STAGES
#define HIPATTN_U8_STAGES 2
#endif

template <bool kU8>
struct BlockRegs;

template <>
struct BlockRegs<false> {
    uint4_t k[2][4];  // [tile][k-step]: K[tile*16 + (lane&15)][kg*32 + i*8 .. +8]
    uint4_t v[8];     // [j = tile*4 + r]: V[tile*16 + kg*4 + r][(lane&15)*8 .. +8]
};

template <>
struct BlockRegs<true> {
    uint2_t k[2][4];  // 8 bytes each
    uint2_t v[8];
    // (scale, zp) of one token: lane (i = lane & 15, kg) holds those of the K row (i < 8) or V row
    // (i >= 8) of token j = i & 7 of its 16-lane row, i.e. of token (j >> 2) * 16 + kg * 4 + (j & 3);
    // the lanes of the row read them with a DPP row broadcast.  (Loading all eight pairs of K and
    // of V into every lane costs sixteen load instructions and 32 registers per block.)
    float2 sz;
};

// A bf16 block turned into fp16 operands in its registers (fp16 queries on a bf16 cache: rounding the queries to
// bf16's eight bits instead costs the decode rows their 2e-3).  bf16 -> fp16 is exact inside fp16's range; beyond it
// the conversion (towards zero) stops at the largest finite fp16 number.
__device__ __forceinline__ uint32_t bf16x2_to_f16x2(uint32_t w) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u)));
}
__device__ __forceinline__ void bf16_block_to_f16(BlockRegs<false>& b) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) b.k[t][i][e] = bf16x2_to_f16x2(b.k[t][i][e]);
#pragma unroll
    for (int j = 0; j < 8; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) b.v[j][e] = bf16x2_to_f16x2(b.v[j][e]);
}

// value of lane kLane of the caller's 16-lane row (v_mov_b32 row_newbcast, folded into the consumer where possible)
template <int kLane>
__device__ __forceinline__ float row_broadcast(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + kLane, 0xf, 0xf, false));
}

// kb[t] / vb[t]: the first row of the unit's 16-token tile t in the key / value cache (one block of
// 32 tokens: kb[1] is sixteen rows behind kb[0]; blocks of 16: two blocks).  Head size kHD: a K row
// is read in kHD / 32 pieces per lane, a V row by the kHD / 8 lanes that have a piece of it.
template <bool kU8, int kHD = kD, int kBlk = kBS>
__device__ __forceinline__ void load_block(BlockRegs<kU8>& b, const uint8_t* const (&kb)[2], const uint8_t* const (&vb)[2],
                                           int n16, int kg) {
    if constexpr (!kU8) {
        constexpr int kRow = 2 * kHD;
        // (with blocks of 32 both tiles are addressed from the block's first row: one base register)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int i = 0; i < kHD / 32; i++)
                b.k[t][i] = kBlk == 32 ? *(const uint4_t*)(kb[0] + (t * 16 + n16) * kRow + kg * (kHD / 2) + i * 16)
                                       : *(const uint4_t*)(kb[t] + n16 * kRow + kg * (kHD / 2) + i * 16);
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (kHD == 128 || n16 * 8 < kHD)
                    b.v[t * 4 + r] = kBlk == 32 ? *(const uint4_t*)(vb[0] + (t * 16 + kg * 4 + r) * kRow + n16 * 16)
                                                : *(const uint4_t*)(vb[t] + (kg * 4 + r) * kRow + n16 * 16);
                else
                    b.v[t * 4 + r] = (uint4_t){0u, 0u, 0u, 0u};
            }
    } else {
        constexpr int kRow = kHD + 8;
        // a lane's K bytes are kHD / 4 consecutive ones of a row, in pieces of eight; its V bytes the
        // eight of its columns, when the head has them
        const bool v_cols = kHD == 128 || n16 * 8 < kHD;
        if constexpr (kBlk == 32) {  // both tiles from the block's first row
            const uint8_t* const kbase = kb[0];
            const uint8_t* const vbase = vb[0];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < kHD / 32; i++)
                    b.k[t][i] = *(const uint2_t*)(kbase + (t * 16 + n16) * kRow + 8 + kg * (kHD / 4) + i * 8);
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int tok = t * 16 + kg * 4 + r;
                    if (v_cols)
                        b.v[t * 4 + r] = *(const uint2_t*)(vbase + tok * kRow + 8 + n16 * 8);
                    else
                        b.v[t * 4 + r] = (uint2_t){0u, 0u};
                }
            {
                const int j = n16 & 7, tok = (j >> 2) * 16 + kg * 4 + (j & 3);
                b.sz = *(const float2*)((n16 < 8 ? kbase : vbase) + tok * kRow);
            }
        } else {  // a block per tile
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < kHD / 32; i++)
                    b.k[t][i] = *(const uint2_t*)(kb[t] + n16 * kRow + 8 + kg * (kHD / 4) + i * 8);
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (v_cols)
                        b.v[t * 4 + r] = *(const uint2_t*)(vb[t] + (kg * 4 + r) * kRow + 8 + n16 * 8);
                    else
                        b.v[t * 4 + r] = (uint2_t){0u, 0u};
                }
            {
                const int j = n16 & 7, row = kg * 4 + (j & 3);
                // One of four tile bases per lane, put together arithmetically: a per-lane index into
                // (or a select among the elements of) the arrays would move them to scratch memory.
                const uintptr_t k0 = (uintptr_t)kb[0], k1 = (uintptr_t)kb[1], v0 = (uintptr_t)vb[0], v1 = (uintptr_t)vb[1];
                const uintptr_t second = (uintptr_t)(j >> 2), value = (uintptr_t)(n16 >> 3);
                const uintptr_t in_k = k0 + second * (k1 - k0), in_v = v0 + second * (v1 - v0);
                b.sz = *(const float2*)(in_k + value * (in_v - in_k) + (uintptr_t)(row * kRow));
            }
        }
    }
}

// The same for a head size below kHD: rows are `row` bytes apart; koff[i] is this lane's offset of K
// piece i inside a tile -- a piece past the end of the row is pointed at the row's first piece, which
// is valid memory and meets zeros in the query operand -- and the lanes whose V columns do not exist
// (v_ok false) get zeros.  voff: the lane's offset of its first V row's piece.  u8 rows: the payload
// behind eight bytes of scale and zero-point, pieces of eight bytes.
template <bool kU8, int kHD, int kBlk>
__device__ __forceinline__ void load_block_padded(BlockRegs<kU8>& b, const uint8_t* const (&kb)[2], const uint8_t* const (&vb)[2],
                                                  int row, const int (&koff)[kHD / 32], int voff, bool v_ok, int n16, int kg) {
    using Piece = typename std::conditional<kU8, uint2_t, uint4_t>::type;
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint8_t* const kt = kBlk == 32 ? kb[0] + t * 16 * row : kb[t];
#pragma unroll
        for (int i = 0; i < kHD / 32; i++) b.k[t][i] = *(const Piece*)(kt + koff[i]);
    }
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint8_t* const vt = kBlk == 32 ? vb[0] + t * 16 * row : vb[t];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            Piece piece = {};
            if (v_ok) piece = *(const Piece*)(vt + voff + r * row);
            b.v[t * 4 + r] = piece;
        }
    }
    if constexpr (kU8) {
        const int j = n16 & 7, at = (kg * 4 + (j & 3)) * row;
        if constexpr (kBlk == 32) {
            b.sz = *(const float2*)((n16 < 8 ? kb[0] : vb[0]) + (j >> 2) * 16 * row + at);
        } else {  // (one of four tile bases per lane, put together arithmetically: see load_block)
            const uintptr_t k0 = (uintptr_t)kb[0], k1 = (uintptr_t)kb[1], v0 = (uintptr_t)vb[0], v1 = (uintptr_t)vb[1];
            const uintptr_t second = (uintptr_t)(j >> 2), value = (uintptr_t)(n16 >> 3);
            const uintptr_t in_k = k0 + second * (k1 - k0), in_v = v0 + second * (v1 - v0);
            b.sz = *(const float2*)(in_k + value * (in_v - in_k) + (uintptr_t)at);
        }
    }
}

struct WaveState {
    float m;          // running max of the scaled scores (log2 domain), per head (lane & 15)
    float l;          // this lane's share of the running sum
    float corr;       // u8 only: this lane's share of sum_j p'_j zp_j
    float4_t acc[8];  // acc[e][r] = O[head][(kg*4 + r)*8 + e]
};

// kTileMask (blocks of 16): `tiles_in` has bit t set when tile t of the unit lies in a block of the
// cache; with blocks of 32 both tiles always do and the argument is ignored.
// kAlibi: slopes holds the ALiBi slopes of the group's query heads (`heads` of them; lane n16 serves head n16),
// and slope * (token - last attended token) joins the scaled score.  The slope is fetched where it is used:
// the loop has no register left to hold it (a constant added to a whole row leaves its softmax alone,
// so the distance may be measured from the row's last attended token instead of its own position).
// A template argument rather than a test of the pointer: the test alone cost the u8 kernel 1.3 %.
template <bool kU8, bool kBf16, int kHD = kD, bool kTileMask = false, bool kAlibi = false>
__device__ __forceinline__ void process_block(WaveState& st, BlockRegs<kU8>& b, const typename Op16<kBf16>::vec8 (&qf)[4], float sumq,
                                              float c, int tok_base, int j0, int ctx, int kg, int tiles_in = 3,
                                              const float* slopes = nullptr, int heads = 0) {
    const int tiles = kTileMask ? tiles_in : 3;
    // ---- S^T = K Q^T : two tiles of 16 tokens x 16 heads
    float4_t s[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
        s[t] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kHD / 32; i++) {
            typename Op16<kBf16>::vec8 a;
            if constexpr (!kU8) {
                a = Op16<kBf16>::from_bits(b.k[t][i]);
            } else {
                uint4_t w;
                w[0] = bytes_to_biased_half2(b.k[t][i][0], 0x04010400u);
                w[1] = bytes_to_biased_half2(b.k[t][i][0], 0x04030402u);
                w[2] = bytes_to_biased_half2(b.k[t][i][1], 0x04010400u);
                w[3] = bytes_to_biased_half2(b.k[t][i][1], 0x04030402u);
                a = Op16<kBf16>::from_bits(w);
            }
            s[t] = Op16<kBf16>::mma(a, qf[i], s[t]);
        }
    }
    // ---- mask, scale, online softmax.  Lane holds tokens tok_base + t*16 + kg*4 + r.
    float sv[8];
    float mloc = -INFINITY;
    // u8: this lane's token's scale, zero-point plus byte bias, and their product (see BlockRegs)
    float sz_scale = 0.0f, sz_zero = 0.0f, sz_prod = 0.0f;
    const bool partial = (tok_base < j0) || (tok_base + kUnit > ctx) || tiles != 3;  // wavefront-uniform
    if constexpr (kU8) {
        sz_scale = b.sz.x;
        sz_zero = b.sz.y + kByteBias;
        if (partial) {
            // Rows outside the attended range may hold anything (never-written cache memory): their
            // probability is exactly zero, and their scale and zero-point are cleared so that
            // 0 * NaN cannot occur.
            const int j = ((int)threadIdx.x & 7), tok = tok_base + (j >> 2) * 16 + kg * 4 + (j & 3);
            if (!(tok >= j0 && tok < ctx && ((tiles >> (j >> 2)) & 1))) sz_scale = sz_zero = 0.0f;
        }
        sz_prod = sz_scale * sz_zero;
    }
    auto dequant_score = [&](auto jc, float x) {
        constexpr int j = decltype(jc)::value;
        return fmaf(row_broadcast<j>(sz_scale), x, -(row_broadcast<j>(sz_prod) * sumq));
    };
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = t * 4 + r;
            const int tok = tok_base + t * 16 + kg * 4 + r;
            float x = s[t][r];
            if constexpr (kU8) {
                switch (j) {
                    case 0: x = dequant_score(std::integral_constant<int, 0>{}, x); break;
                    case 1: x = dequant_score(std::integral_constant<int, 1>{}, x); break;
                    case 2: x = dequant_score(std::integral_constant<int, 2>{}, x); break;
                    case 3: x = dequant_score(std::integral_constant<int, 3>{}, x); break;
                    case 4: x = dequant_score(std::integral_constant<int, 4>{}, x); break;
                    case 5: x = dequant_score(std::integral_constant<int, 5>{}, x); break;
                    case 6: x = dequant_score(std::integral_constant<int, 6>{}, x); break;
                    default: x = dequant_score(std::integral_constant<int, 7>{}, x); break;
                }
            }
            x = (tok >= j0 && tok < ctx && ((tiles >> t) & 1)) ? x * c : -INFINITY;
            sv[j] = x;
            if constexpr (!kAlibi) mloc = fmaxf(mloc, x);
        }
    if constexpr (kAlibi) {
        const int n16 = (int)threadIdx.x & 15;
        const float slope = *(const volatile float*)(slopes + (n16 < heads ? n16 : 0)) * kLog2e;
        const float first = (float)(tok_base + kg * 4 - (ctx - 1));
#pragma unroll
        for (int j = 0; j < 8; j++) {
            sv[j] = fmaf(slope, first + (float)((j >> 2) * 16 + (j & 3)), sv[j]);
            mloc = fmaxf(mloc, sv[j]);
        }
    }
    mloc = max_over_rows(mloc);
    const float m_new = fmaxf(st.m, mloc);  // finite: every processed block holds an attended token
    const float alpha = fast_exp2(st.m - m_new);
    st.m = m_new;
    // Rows outside the attended range may hold anything (never-written cache memory): their
    // probability is exactly zero, and fp16 V rows are cleared so that 0 * NaN cannot occur.
    if constexpr (!kU8) {
        if (partial) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int tok = tok_base + (j >> 2) * 16 + kg * 4 + (j & 3);
                if (!(tok >= j0 && tok < ctx && ((tiles >> (j >> 2)) & 1))) b.v[j] = (uint4_t){0u, 0u, 0u, 0u};
            }
        }
    }
    typename Op16<kBf16>::vec8 pf;
    float lsum = 0.0f, csum = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        float pj = fast_exp2(sv[j] - m_new);
        lsum += pj;
        if constexpr (kU8) {
            float vs, vz;  // scale and zero-point (plus bias) of V's token j: lanes 8 + j of the row
            switch (j) {
                case 0: vs = row_broadcast<8>(sz_scale); vz = row_broadcast<8>(sz_zero); break;
                case 1: vs = row_broadcast<9>(sz_scale); vz = row_broadcast<9>(sz_zero); break;
                case 2: vs = row_broadcast<10>(sz_scale); vz = row_broadcast<10>(sz_zero); break;
                case 3: vs = row_broadcast<11>(sz_scale); vz = row_broadcast<11>(sz_zero); break;
                case 4: vs = row_broadcast<12>(sz_scale); vz = row_broadcast<12>(sz_zero); break;
                case 5: vs = row_broadcast<13>(sz_scale); vz = row_broadcast<13>(sz_zero); break;
                case 6: vs = row_broadcast<14>(sz_scale); vz = row_broadcast<14>(sz_zero); break;
                default: vs = row_broadcast<15>(sz_scale); vz = row_broadcast<15>(sz_zero); break;
            }
            pj *= vs;
            Op16<kBf16>::set(pf, j, pj);
            csum = fmaf(Op16<kBf16>::get(pf, j), vz, csum);
        } else {
            Op16<kBf16>::set(pf, j, pj);
        }
    }
    st.l = st.l * alpha + lsum;
    if constexpr (kU8) st.corr = st.corr * alpha + csum;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
        for (int e = 0; e < 8; e++) st.acc[e] *= alpha;
    }
    // ---- O^T += V^T P^T : transpose the lane's 8 tokens x 8 head-dim patch in registers
#pragma unroll
    for (int e = 0; e < 8; e++) {
        uint4_t w;
        if constexpr (!kU8) {
#pragma unroll
            for (int jp = 0; jp < 4; jp++) {
                const uint32_t lo = b.v[2 * jp][e >> 1], hi = b.v[2 * jp + 1][e >> 1];
                w[jp] = (e & 1) ? pack_hi(lo, hi) : pack_lo(lo, hi);
            }
        } else {
            const uint32_t sel = 0x0c000c00u | ((4u + (e & 3)) << 16) | (uint32_t)(e & 3);
#pragma unroll
            for (int jp = 0; jp < 4; jp++)
                w[jp] = bytes_to_biased_half2(b.v[2 * jp][e >> 2], b.v[2 * jp + 1][e >> 2], sel);
        }
        st.acc[e] = Op16<kBf16>::mma(Op16<kBf16>::from_bits(w), pf, st.acc[e]);
    }
}


// Length of one (sequence, kv head) segment on the work line: its blocks plus `switch_cost`
// units that stand for the time a wavefront loses when it starts on a new segment (dependent
// loads of the sequence's lengths, its block table and the queries).  Cutting the line into
// equal pieces then equalises time, not just bytes.
__device__ __forceinline__ int line_units(int nb, int switch_cost) { return nb > 0 ? nb + switch_cost : 0; }

__device__ __forceinline__ void zero_output_row(const PagedParams& p, int token) {
    const int64_t n = (int64_t)p.num_heads_q * p.head_dim, o0 = (int64_t)token * n;
    for (int64_t e = 0; e < n; e++) {
        if (p.out_dtype == HIPATTN_F32)
            ((float*)p.out)[o0 + e] = 0.0f;
        else
            ((uint16_t*)p.out)[o0 + e] = 0;
    }
}

// How the work line [0, total) is cut into pieces.  Pieces 0 .. W-1 are the static ones, one per
// wavefront, and share the first three quarters of the line equally; pieces W .. W+P-1 share the
// last quarter and are handed out on demand (an atomic counter), so wavefronts that run faster
// -- older ones win the arbitration for the memory pipeline, some XCDs see more bandwidth --
// take more of them and all wavefronts finish together.
struct Line {
    int64_t total, t_static, t_dyn;
    int W, P;
    __device__ __forceinline__ Line(int64_t total_, int W_, int P_) : total(total_), W(W_), P(P_) {
        t_dyn = P_ > 0 ? total_ / 4 : 0;
        t_static = total_ - t_dyn;
    }
    // first line unit of piece id (id may be W + P: the end of the line)
    __device__ __forceinline__ int64_t begin(int id) const {
        if (id <= W) return (int64_t)id * t_static / W;
        return t_static + (int64_t)(id - W) * t_dyn / P;
    }
    // the (non-empty) piece that holds line unit pos, 0 <= pos < total
    __device__ __forceinline__ int piece_at(int64_t pos) const {
        if (pos < t_static) return (int)(((pos + 1) * W - 1) / t_static);
        return W + (int)(((pos - t_static + 1) * P - 1) / t_dyn);
    }
};

// Wavefronts of `waves` that get a piece of a line of `total` units (p.few_waves == 0: all of them).  A small batch on all of
// them is bound by combining what they leave: every piece of a segment is one more partial for the merge.  So pieces
// are eight units or more, except that half of the ordinary count of wavefronts and two per segment are never too many
// (p.few_waves), and none is empty; beyond one per compute unit only whole numbers of them per compute unit (17 % more
// time with 1,088 than with 1,024).  One sequence of 778 tokens: 13.7 us with 1,024 wavefronts, 11.7 with the 240 this gives
// it (64: 12.9); of 4,000: 14.3 / 13.1 with 1,024 / 512; u8, 16 sequences of 300 (128 segments): 22.5 / 17.1 with 1,536 / 512.
__host__ __device__ __forceinline__ int working_waves(const PagedParams& p, int64_t total, int waves) {
    if (p.few_waves == 0) return waves;
    const int eighth = total >= 8 * (int64_t)waves ? waves : (int)(total >> 3);  // (no division: it took 0.3 us of both kernels)
    int n = eighth > p.few_waves ? eighth : p.few_waves;
    if (n > 256) n = (n + 128) & ~255;
    if (n > 1024) n &= ~511;  // (five wavefronts to a compute unit's four SIMDs: u8, 79 sequences of 40 to 335, 24.8 us with 1,280, 24.0 with 1,024)
    if (n > waves) n = waves;
    if (n > total) n = total > 256 ? (int)total & ~255 : (int)total;
    return n;
}

// eight consecutive output elements, one 16-byte store for the 16-bit types
__device__ __forceinline__ void store_out8(void* out, int64_t elem, int dtype, const float (&o)[8]) {
    if (dtype == HIPATTN_F32) {
        float* po = (float*)out + elem;
        *(float4*)(po) = make_float4(o[0], o[1], o[2], o[3]);
        *(float4*)(po + 4) = make_float4(o[4], o[5], o[6], o[7]);
        return;
    }
    uint4_t w;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t lo = dtype == HIPATTN_F16 ? float_to_f16_bits(o[2 * i]) : float_to_bf16_bits(o[2 * i]);
        const uint32_t hi = dtype == HIPATTN_F16 ? float_to_f16_bits(o[2 * i + 1]) : float_to_bf16_bits(o[2 * i + 1]);
        w[i] = lo | (hi << 16);
    }
    *(uint4_t*)((uint16_t*)out + elem) = w;
}

// ---- partial results that another wavefront of the same launch reads ------------------------
// The compute units of the device sit behind eight L2 caches that are not kept coherent for
// ordinary accesses.  Partials, and the flags that announce them, therefore go through agent-scope
// relaxed atomic accesses (write-through stores, loads that do not take a stale line): no fence,
// which would write back and invalidate whole L2 caches while the kernel streams through them.
// Order is kept by hand: a producer waits for its stores (s_waitcnt vmcnt(0)) before it raises
// the flag, a consumer reads the partial only after it has seen the flag.
//
// Layout of such a partial (fused_merge; the merge kernel's partials keep theirs): the wavefront that
// combines has the lane layout of the one that produced, so a lane's 32 accumulator values and its
// head's (max, sum) travel as seventeen pairs of floats, pair j of active lane a (a = kg * G + head,
// 4 G of them) at pair index j * 4 G + a of the slot.  One store instruction then writes 4 G x 8
// contiguous bytes -- whole cache lines from four query heads per kv head on -- which matters because a
// write-through store of part of a line is a read-modify-write at the memory (4-byte stores, sixteen
// lines per instruction, cost configuration 3's kernel 20 us).
constexpr int kPartPairs = 17;  // per active lane: 16 pairs of outputs, then (max, sum)
__device__ __forceinline__ void agent_store2(float* p, float x, float y) {
    const unsigned long long v = (unsigned long long)__float_as_uint(x) | ((unsigned long long)__float_as_uint(y) << 32);
    __hip_atomic_store((unsigned long long*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_load2(const float* p, float& x, float& y) {
    const unsigned long long v = __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    x = __uint_as_float((uint32_t)v);
    y = __uint_as_float((uint32_t)(v >> 32));
}
__device__ __forceinline__ void stores_done() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// The wavefront that holds the LAST units of a segment which other pieces worked on too combines
// the partials of all of them (its own among them, left in the workspace like the others) when its
// own piece is done: a piece meets such a segment only as the first of its run, so it has at most
// one to combine, and the pieces it waits for have lower numbers, i.e. were dispatched before it.
// Lane (head n16, kg) owns head-dim (kg*4 + r)*8 + e of its head, as in the accumulators.
// Waiting is bounded (kMergeSpinLimit polls of about a microsecond each): a flag that never comes --
// which a consistent plan cannot produce -- leaves the rows unwritten instead of a hung wavefront.
constexpr int kMergeSpinLimit = 1 << 22;
struct MergeArgs {
    float* part_out;
    float* part_ml;
    uint64_t* part_flag;
    unsigned long long merge_tag;
    void* out;
    int out_dtype, num_heads_q, num_heads_kv, head_dim;
    const float* sinks;
};
template <int kHD, bool kPad>
__device__ __forceinline__ void merge_in_kernel(const MergeArgs& p, const Line& line, int s, int h, int token,
                                                int id_first, int id_last, int lane) {
    const int Hkv = p.num_heads_kv, G = p.num_heads_q / p.num_heads_kv;
    const int head_dim = kPad ? p.head_dim : kHD;
    const int n16 = lane & 15, kg = lane >> 4;
    // flags of the other pieces: lane i polls piece id_first + i (64 at a time)
    for (int id0 = id_first; id0 < id_last; id0 += 64) {
        const int id = id0 + lane;
        const bool have = id < id_last && line.begin(id) < line.begin(id + 1);  // (empty pieces leave nothing)
        unsigned long long* flag = (unsigned long long*)p.part_flag + ((int64_t)id + (int64_t)s * Hkv + h);
        bool ready = !have;
        for (int spin = 0; spin < kMergeSpinLimit; spin++) {
            if (!ready) ready = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == p.merge_tag;
            if (__builtin_amdgcn_ballot_w64(!ready) == 0) break;
            __builtin_amdgcn_s_sleep(2);
        }
        if (__builtin_amdgcn_ballot_w64(!ready) != 0) return;
        // taken: a replay of a captured call comes with the same tag and must not see this flag again
        if (have) __hip_atomic_store(flag, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    float m_run = -INFINITY, l_run = 0.0f;
    float4_t acc[8];
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] = (float4_t){0.f, 0.f, 0.f, 0.f};
    const bool mine = n16 < G;
    // two pieces at a time, every load of the two issued before the first is used: the merge is a chain
    // of memory round trips at the very end of the kernel, and four at a time make the register allocator spill
    for (int id0 = id_first; id0 <= id_last; id0 += 2) {
        float mw[2], lw[2];
        float4_t part[2][8];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int id = id0 + u;
            mw[u] = -INFINITY;
            lw[u] = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) part[u][e] = (float4_t){0.f, 0.f, 0.f, 0.f};
            if (mine && id <= id_last && line.begin(id) < line.begin(id + 1)) {
                const int64_t slot = (int64_t)id + (int64_t)s * Hkv + h;
                const float* rec = p.part_out + (slot * kPartPairs * 4 * G + (kg * G + n16)) * 2;
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int e2 = 0; e2 < 4; e2++) {
                        float x, y;
                        agent_load2(rec + (r * 4 + e2) * 8 * G, x, y);
                        part[u][2 * e2][r] = x;
                        part[u][2 * e2 + 1][r] = y;
                    }
                agent_load2(rec + 16 * 8 * G, mw[u], lw[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const float m_new = fmaxf(m_run, mw[u]);
            const float rescale = (m_run == -INFINITY) ? 0.0f : fast_exp2(m_run - m_new);
            const float f = (mw[u] == -INFINITY) ? 0.0f : fast_exp2(mw[u] - m_new);
            l_run = l_run * rescale + f * lw[u];
#pragma unroll
            for (int e = 0; e < 8; e++) acc[e] = acc[e] * rescale + part[u][e] * f;
            m_run = m_new;
        }
    }
    if (!mine) return;
    if (p.sinks != nullptr && l_run > 0.0f) l_run += fast_exp2(p.sinks[h * G + n16] * kLog2e - m_run);
    const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int d0 = (kg * 4 + r) * 8;
        if ((kPad || kHD < 128) && d0 >= head_dim) continue;
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = acc[e][r] * inv;
        store_out8(p.out, ((int64_t)token * p.num_heads_q + h * G + n16) * head_dim + d0, p.out_dtype, o);
    }
}

// Pure decode batches of up to kSelfPlanMaxRows rows need no prologue launch: every wavefront works
// out the schedule for itself (one record per row into LDS, lane-parallel, and a wavefront scan for
// the prefix sums), which is shorter than the chain of dependent global loads through a plan another
// kernel left behind, and the wavefront that is about to read the last cache block of a (row, kv
// head) first writes that row's new K and V rows into it -- the operator's cache write, done by
// the only wavefront that needs its result during this call.  Wavefront 0 leaves the plan in the
// workspace for the merge kernel.
constexpr int kSelfPlanMaxRows = 256;

// kWaves wavefronts to a workgroup.  1 is the ordinary launch.  With 8 a workgroup owns a compute
// unit's whole register file: `gridDim.x` workgroups then keep exactly that many compute units and
// leave the others free for a kernel that runs beside this one.
// kHD, kBlk: head size (128 or 64) and cache block size (32, 16, or 0: a larger power of two); the self-planning form and the
// eight-wavefront form exist for head size 128 only (the eight-wavefront form also for 16-bit caches at the
// head sizes between 64 and 128, kPad), the self-planning form on blocks of 32 or 16 only.
// kPad: the call's head size (p.head_dim, a multiple of 8) may be smaller than kHD: the missing columns of
// Q are zeros and those of V are not read.
template <bool kU8, bool kBf16, int kWaves, bool kSelfPlan = false, int kHD = kD, int kBlk = kBS, bool kPad = false, bool kAlibi = false, bool kHalfFromBf16 = false>
__device__ __forceinline__ void paged_decode_body(const PagedParams& p, const KvWriteParams& wp, int do_write, int workgroup) {
    // kHalfFromBf16: the cache holds bf16, the operands are fp16 (fp16 queries): blocks are converted as they arrive
    static_assert(!kHalfFromBf16 || (!kU8 && !kBf16 && kWaves == 1 && !kSelfPlan && kHD == 128 && !kPad && !kAlibi), "bf16 blocks as fp16 operands: the ordinary launch at head size 128 only");
    static_assert(!kAlibi || (kWaves == 1 && !kSelfPlan), "the distance bias (p.alibi_slopes) exists in the ordinary launch only");
    // The merge inside the kernel (p.fused_merge) is built into the u8 instantiations only: the 16-bit ones use
    // every register in their loop, and with that code behind the loop the allocator spilled 29 of them.
    constexpr bool kFusedBuilt = kU8;
    static_assert(!(kU8 && kBf16), "u8 caches are dequantised to fp16 operands");
    static_assert(!kPad || (!kSelfPlan && (kWaves == 1 || (kHD == 128 && !kU8))), "padded head sizes: no self-planning form; eight wavefronts for 16-bit caches in the head-128 build");
    static_assert(kHD == 128 || (!kSelfPlan && kWaves == 1), "head size 64 has the ordinary launch only");
    static_assert((kHD == 64 || kHD == 128) && (kBlk == 16 || kBlk == 32 || kBlk == 0), "head size 64 or 128, blocks of 16, 32 or more");
    // kBlk == 0: any larger power of two (p.block_size); a block then holds several units, one after the other
    static_assert(kBlk != 0 || !kSelfPlan, "larger blocks: no self-planning form");
    constexpr int kEntries = kBlk == 16 ? 2 : 1;  // block-table entries per unit
    constexpr int kTileBlk = kBlk == 16 ? 16 : 32;  // how a unit's two tiles lie: a block each, or sixteen rows apart
    const int blk = kBlk ? kBlk : p.block_size;
    const int sub_mask = kBlk ? 0 : (p.block_size >> 5) - 1;  // kBlk == 0: unit u is part (u & sub_mask) of its block
    static_assert(!kSelfPlan || kWaves == 1, "a wavefront that plans for itself is a workgroup of its own");
    const int w = kWaves == 1 ? workgroup : workgroup * kWaves + (int)(threadIdx.x >> 6);
    const int lane = kWaves == 1 ? threadIdx.x : (threadIdx.x & 63), n16 = lane & 15, kg = lane >> 4;
    const int Hkv = p.num_heads_kv, G = p.num_heads_q / p.num_heads_kv;
    const float c = p.scale * kLog2e;
    __shared__ DecodeRange plan_rec[kSelfPlan ? kSelfPlanMaxRows : 1];
    __shared__ int plan_prefix[kSelfPlan ? kSelfPlanMaxRows + 1 : 1];
    if constexpr (kSelfPlan) {
        int carry = 0;
        for (int base = 0; base < p.num_rows; base += 64) {
            const int i = base + lane;
            DecodeRange rg;
            int units = 0;
            if (i < p.num_rows) {
                rg = decode_range(p, i);
                units = line_units(rg.nb, p.switch_cost);
                plan_rec[i] = rg;
            }
            int scan = units;  // inclusive scan over the wavefront
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int up = __shfl_up(scan, d, 64);
                if (lane >= d) scan += up;
            }
            if (i < p.num_rows) {
                plan_prefix[i] = carry + scan - units;
                if (w == 0) {  // for the merge kernel
                    ((DecodeRange*)p.seq_info)[i] = rg;
                    p.blk_prefix[i] = carry + scan - units;
                    if (rg.empty_row) zero_output_row(p, rg.token);
                }
            }
            carry += __shfl(scan, 63, 64);
        }
        if (lane == 0) {
            plan_prefix[p.num_rows] = carry;
            if (w == 0) p.blk_prefix[p.num_rows] = carry;
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the records are in LDS (the wavefront is the whole workgroup)
        __builtin_amdgcn_wave_barrier();
    }
    auto prefix_at = [&](int i) -> int {
        if constexpr (kSelfPlan)
            return plan_prefix[i];
        else
            return p.blk_prefix[i];
    };
    const int64_t total = (int64_t)prefix_at(p.num_rows) * Hkv;
    if (total <= 0) return;
    // eight to a workgroup: the plan has chosen how many of the launched wavefronts work
    const int num_waves = working_waves(p, total, kWaves == 1 ? p.num_waves : p.plan_waves[0]);
    if (w >= num_waves) return;
    const Line line(total, num_waves, p.dyn_pieces);

    constexpr int64_t kRowBytesBuilt = kU8 ? (kHD + 8) : (2 * kHD);
    const int head_dim = kPad ? p.head_dim : kHD;                       // (a constant unless kPad)
    const int64_t kRowBytes = kPad ? (kU8 ? p.head_dim + 8 : 2 * p.head_dim) : kRowBytesBuilt;
    const int64_t block_stride = (int64_t)(Hkv / p.kv_share) * blk * kRowBytes;  // (kv_share: see PagedParams)
    // kPad: this lane's K piece offsets, V offset and whether its V columns exist
    int koff[kHD / 32];
    int voff = 0;
    bool v_ok = true;
    if constexpr (kPad) {
#pragma unroll
        for (int i = 0; i < kHD / 32; i++) {
            const int first = kg * (kHD / 4) + i * 8;  // first of the piece's eight columns
            koff[i] = n16 * (int)kRowBytes + (kU8 ? 8 + (first < head_dim ? first : 0) : (first < head_dim ? first * 2 : 0));
        }
        voff = kg * 4 * (int)kRowBytes + (kU8 ? 8 + n16 * 8 : n16 * 16);
        v_ok = n16 * 8 < head_dim;
    }

    // The static piece first, then dynamic pieces for as long as there are any.  The ticket for
    // the next dynamic piece is drawn before the current piece is worked on, so its latency is hidden.
    // Tickets come from one counter per group of wavefronts (a single counter would serialise
    // thousands of same-address atomics); group g owns the dynamic pieces g, g + groups, ...
    // A group mixes wavefronts of every XCD and of both dispatch halves (w / 8 mod groups).
    const int group = (w >> 3) % p.dyn_groups;
    int piece = w;
    int merge_seg = -1;  // (fused_merge) the segment this piece has to combine, as sequence * kv heads + kv head
    for (;;) {
    int ticket_lane0 = 0;
    if (p.dyn_pieces > 0 && lane == 0) ticket_lane0 = atomicAdd(p.dyn_counter + group, 1);
    int64_t L = line.begin(piece);
    const int64_t L_end = line.begin(piece + 1);
    int s = 0;
    if (L < L_end) {
        if constexpr (kSelfPlan) {  // the last row whose prefix is <= L / Hkv (the prefix is monotone)
            const int x = (int)(L / Hkv);
            int cnt = 0;
            for (int base = 0; base < p.num_rows; base += 64) {
                const int i = base + lane;
                cnt += __builtin_popcountll(__builtin_amdgcn_ballot_w64(i < p.num_rows && plan_prefix[i] <= x));
            }
            s = max(cnt - 1, 0);
        } else {
            s = locate_sequence(p.blk_prefix, p.num_rows, (int)(L / Hkv), lane);
        }
    }

    while (L < L_end) {
        while (s + 1 < p.num_rows && (int64_t)prefix_at(s + 1) * Hkv <= L) s++;  // next row with blocks
        DecodeRange rg;
        if constexpr (kSelfPlan)
            rg = plan_rec[s];
        else
            rg = ((const DecodeRange*)p.seq_info)[s];
        const int nb = rg.nb;
        if (nb <= 0) break;  // cannot happen for a consistent plan; never loop forever
        const int seglen = nb + p.switch_cost;
        const int64_t seq_L0 = (int64_t)prefix_at(s) * Hkv;
        const int h = (int)((L - seq_L0) / seglen);
        const int64_t seg_B0 = seq_L0 + (int64_t)h * seglen + p.switch_cost;  // line position of the segment's block 0
        const int64_t seg_L1 = seg_B0 + nb;                        // end of the segment
        const int64_t from = max(L, seg_B0), to = min(L_end, seg_L1);
        if (from >= to) {  // the piece ends inside the switch-cost units: no block of this segment is ours
            L = to;
            continue;
        }
        const int b_rel = (int)(from - seg_B0);
        const int n = (int)(to - from);  // blocks of this segment in this piece
        const bool whole = (n == nb);
        L = from;
        // the segment ends here and began in an earlier piece: this piece combines it when it is done
        // (one scalar carried through the loop; the rest is worked out again then)
        if constexpr (kFusedBuilt) {
            if (p.fused_merge && !whole && b_rel + n == nb) merge_seg = s * Hkv + h;
        }
        const int lb0 = rg.j0 / kUnit + b_rel;          // first unit of 32 tokens
        // (kBlk == 0: the table is indexed by the block of the absolute unit, lb0 + ... >> log2(units per block))
        const int32_t* table = p.block_indices + rg.table_begin + (kBlk ? lb0 * kEntries : 0);
        // table entries from there on that hold attended tokens (the row's table may end with them)
        const int entries = (rg.ctx + blk - 1) / blk - (kBlk ? lb0 * kEntries : 0);
        const int h_kv = p.kv_share == 1 ? h : h / p.kv_share;  // the kv head whose rows this segment reads
        const int64_t head_off = (int64_t)h_kv * blk * kRowBytes;
        const int sub_shift = kBlk ? 0 : __builtin_ctz(p.block_size >> 5);

        if constexpr (kSelfPlan) {
            // The new tokens of this call whose cache rows this piece is about to read go into the cache
            // first: the row's own token (in the segment's last block) and, when its sequence
            // contributes several tokens to the batch, the tokens ahead of it.  The same wavefront
            // stores and then loads, and the stores are waited for below; a token that several rows
            // attend is written by each of their wavefronts with the same bytes.
            if (do_write && rg.write_pos >= 0) {
                const int q_lo = max(rg.new_begin, lb0 * kUnit), q_hi = min(rg.write_pos, (lb0 + n) * kUnit - 1);
                for (int q = q_lo; q <= q_hi; q++) {  // (wave-uniform; one pass for a decode row)
                    const int pb_new = p.block_indices[rg.table_begin + q / blk];
                    if (pb_new >= 0 && pb_new < p.num_blocks)
                        kv_cache_write_pair128(wp, rg.token - (rg.write_pos - q), h_kv, pb_new, q, lane);
                }
                if (q_lo <= q_hi) __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the rows have reached the cache
            }
        }
        // Q^T operand: lane (head n16, kg) holds Q[head][kg * kHD/4 + i*8 .. +8]; padding heads are zero
        typename Op16<kBf16>::vec8 qf[4];
        float sumq = 0.0f;
        {
            const int64_t qrow = ((int64_t)rg.token * p.num_heads_q + (int64_t)h * G + n16) * head_dim;
#pragma unroll
            for (int i = 0; i < kHD / 32; i++) {
                if (n16 < G && (!kPad || kg * (kHD / 4) + i * 8 < head_dim)) {
                    qf[i] = load_q8<kBf16>(p.q, qrow + kg * (kHD / 4) + i * 8, p.q_dtype);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) Op16<kBf16>::set(qf[i], e, 0.0f);
                }
                if constexpr (kU8) {
#pragma unroll
                    for (int e = 0; e < 8; e++) sumq += Op16<kBf16>::get(qf[i], e);
                }
            }
            if constexpr (kU8) {
                sumq += __shfl_xor(sumq, 16, 64);
                sumq += __shfl_xor(sumq, 32, 64);
            }
        }

        WaveState st;
        st.m = -INFINITY;
        st.l = 0.0f;
        st.corr = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) st.acc[e] = (float4_t){0.f, 0.f, 0.f, 0.f};
        const float* const slopes = kAlibi ? p.alibi_slopes + h * G : nullptr;  // ALiBi, this group's heads

        // units in groups of 64 table entries: one vector load fetches the group's block-table entries
        constexpr int kGroup = 64 / kEntries;
        for (int g0 = 0; g0 < n; g0 += kGroup) {
            const int gn = min(kGroup, n - g0);
            const int my_entry = kBlk ? g0 * kEntries + lane : (lb0 + g0 + lane) >> sub_shift;
            const int my_pb = (lane < gn * kEntries && my_entry < entries) ? table[my_entry] : -1;
            // which tiles of unit i were issued (0: none, the unit is skipped); never reads outside the cache
            auto issue = [&](BlockRegs<kU8>& regs, int i) -> int {
                if constexpr (kEntries == 1) {
                    const int pb = __builtin_amdgcn_readlane(my_pb, i);
                    if (pb < 0 || pb >= p.num_blocks) return 0;
                    int64_t off = (int64_t)pb * block_stride + head_off;
                    if constexpr (kBlk == 0) off += (int64_t)((lb0 + g0 + i) & sub_mask) * (kUnit * kRowBytes);
                    const uint8_t* const kb[2] = {p.key_cache + off, p.key_cache + off + 16 * kRowBytes};
                    const uint8_t* const vb[2] = {p.value_cache + off, p.value_cache + off + 16 * kRowBytes};
                    if constexpr (kPad)
                        load_block_padded<kU8, kHD, kTileBlk>(regs, kb, vb, (int)kRowBytes, koff, voff, v_ok, n16, kg);
                    else
                        load_block<kU8, kHD, kTileBlk>(regs, kb, vb, n16, kg);
                    return 3;
                } else {
                    const int pb0 = __builtin_amdgcn_readlane(my_pb, 2 * i), pb1 = __builtin_amdgcn_readlane(my_pb, 2 * i + 1);
                    // A tile counts only if it holds an attended token: a unit whose one valid block lies wholly
                    // ahead of the window (or behind the context) is skipped like a unit without blocks, so that
                    // every processed unit has a finite score.
                    const int tok0 = (lb0 + g0 + i) * kUnit;
                    const int ok = (pb0 >= 0 && pb0 < p.num_blocks && tok0 + 16 > rg.j0 && tok0 < rg.ctx ? 1 : 0) |
                                   (pb1 >= 0 && pb1 < p.num_blocks && tok0 + 32 > rg.j0 && tok0 + 16 < rg.ctx ? 2 : 0);
                    if (ok == 0) return 0;
                    // a tile without a block is read from the other tile's block: valid memory, and masked
                    const int64_t off0 = (int64_t)((ok & 1) ? pb0 : pb1) * block_stride + head_off;
                    const int64_t off1 = (int64_t)((ok & 2) ? pb1 : pb0) * block_stride + head_off;
                    const uint8_t* const kb[2] = {p.key_cache + off0, p.key_cache + off1};
                    const uint8_t* const vb[2] = {p.value_cache + off0, p.value_cache + off1};
                    if constexpr (kPad)
                        load_block_padded<kU8, kHD, kTileBlk>(regs, kb, vb, (int)kRowBytes, koff, voff, v_ok, n16, kg);
                    else
                        load_block<kU8, kHD, kTileBlk>(regs, kb, vb, n16, kg);
                    return ok;
                }
            };
            if constexpr (!kU8) {
                // two register stages: block i+1 is in flight while block i is consumed
                BlockRegs<kU8> ra, rb;
                int ok_a = issue(ra, 0), ok_b = 0;
                int i = 0;
                while (i < gn) {
                    ok_b = (i + 1 < gn) ? issue(rb, i + 1) : 0;
                    if constexpr (kHalfFromBf16) bf16_block_to_f16(ra);
                    if (ok_a) process_block<kU8, kBf16, kHD, kEntries != 1, kAlibi>(st, ra, qf, sumq, c, (lb0 + g0 + i) * kUnit, rg.j0, rg.ctx, kg, ok_a, slopes, G);
                    if (i + 1 >= gn) break;
                    ok_a = (i + 2 < gn) ? issue(ra, i + 2) : 0;
                    if constexpr (kHalfFromBf16) bf16_block_to_f16(rb);
                    if (ok_b) process_block<kU8, kBf16, kHD, kEntries != 1, kAlibi>(st, rb, qf, sumq, c, (lb0 + g0 + i + 1) * kUnit, rg.j0, rg.ctx, kg, ok_b, slopes, G);
                    i += 2;
                }
            } else {
                // kStages register stages: blocks i+1 .. i+kStages-1 are in flight while block i is
                // consumed.  (Measured on the 128-sequence u8 workload: two stages 452 us, three 455 us,
                // four spill registers and fall to 629 us.)
                constexpr int kStages = HIPATTN_U8_STAGES;
                BlockRegs<kU8> regs[kStages];
                int ok[kStages];
#pragma unroll
                for (int u = 0; u < kStages - 1; u++) ok[u] = (u < gn) ? issue(regs[u], u) : 0;
                for (int i = 0; i < gn; i += kStages) {
#pragma unroll
                    for (int u = 0; u < kStages; u++) {
                        const int idx = i + u;
                        if (idx >= gn) break;
                        constexpr int kLast = kStages - 1;
                        ok[(u + kLast) % kStages] =
                            (idx + kLast < gn) ? issue(regs[(u + kLast) % kStages], idx + kLast) : 0;
                        if (ok[u]) process_block<kU8, kBf16, kHD, kEntries != 1, kAlibi>(st, regs[u], qf, sumq, c, (lb0 + g0 + idx) * kUnit, rg.j0, rg.ctx, kg, ok[u], slopes, G);
                    }
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
        const int64_t slot = (int64_t)piece + (int64_t)s * Hkv + h;  // unique per (piece, segment)
        if (n16 < G) {
            if (whole && p.sinks != nullptr && l > 0.0f) l += fast_exp2(p.sinks[h * G + n16] * kLog2e - st.m);
            const float inv = whole ? (l > 0.0f ? 1.0f / l : 0.0f) : 1.0f;
            // acc[e][r] is head-dim (kg*4 + r)*8 + e: eight consecutive outputs per r
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float o[8];
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    float v = st.acc[e][r];
                    if constexpr (kU8) v -= corr;
                    o[e] = v * inv;
                }
                const int d0 = (kg * 4 + r) * 8;
                // (rows of the accumulator beyond the head size hold nothing; a fused partial carries them all the same)
                if ((kPad || kHD < 128) && d0 >= head_dim && (whole || !(kFusedBuilt && p.fused_merge))) continue;
                if (whole) {
                    store_out8(p.out, ((int64_t)rg.token * p.num_heads_q + h * G + n16) * head_dim + d0, p.out_dtype, o);
                } else if (kFusedBuilt && p.fused_merge) {
                    float* rec = p.part_out + (slot * kPartPairs * 4 * G + (kg * G + n16)) * 2;
#pragma unroll
                    for (int e2 = 0; e2 < 4; e2++) agent_store2(rec + (r * 4 + e2) * 8 * G, o[2 * e2], o[2 * e2 + 1]);
                } else {
                    float* po = p.part_out + (slot * G + n16) * head_dim + d0;
                    *(float4*)(po) = make_float4(o[0], o[1], o[2], o[3]);
                    *(float4*)(po + 4) = make_float4(o[4], o[5], o[6], o[7]);
                }
            }
            if (kFusedBuilt && !whole && p.fused_merge) {
                agent_store2(p.part_out + (slot * kPartPairs * 4 * G + (kg * G + n16)) * 2 + 16 * 8 * G, st.m, l);
            } else if (!whole && kg == 0) {
                p.part_ml[(slot * G + n16) * 2] = st.m;
                p.part_ml[(slot * G + n16) * 2 + 1] = l;
            }
        }
        if (kFusedBuilt && p.fused_merge && !whole && b_rel + n < nb) {
            // a partial another wavefront will combine: announced once the stores above have completed
            // (no load is in flight at the end of a segment, so the wait is for these stores alone)
            stores_done();
            if (lane == 0)
                __hip_atomic_store((unsigned long long*)p.part_flag + slot, p.merge_tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        L += n;
    }
    if (kFusedBuilt && merge_seg >= 0) {
        stores_done();  // this wavefront's own partial of that segment
        const int ms = merge_seg / Hkv, mh = merge_seg - ms * Hkv;
        DecodeRange mr;
        if constexpr (kSelfPlan)
            mr = plan_rec[ms];
        else
            mr = ((const DecodeRange*)p.seq_info)[ms];
        const int64_t first_unit = (int64_t)prefix_at(ms) * Hkv + (int64_t)mh * (mr.nb + p.switch_cost) + p.switch_cost;
        const MergeArgs ma = {p.part_out, p.part_ml, p.part_flag, p.merge_tag, p.out, p.out_dtype, p.num_heads_q, p.num_heads_kv, p.head_dim, p.sinks};
        merge_in_kernel<kHD, kPad>(ma, line, ms, mh, mr.token, line.piece_at(first_unit), piece, lane);
        merge_seg = -1;
    }
    if (p.dyn_pieces <= 0) break;
    const int next = group + __shfl(ticket_lane0, 0, 64) * p.dyn_groups;
    if (next >= p.dyn_pieces) break;  // this group's share of the line is used up (every wavefront gets here)
    piece = num_waves + next;
    }
}

}  // namespace hipattn
