// The flash kernels of flash_chunk.hpp on dense operands (v13::ScaledDotProductAttention) and, for calls whose
// decode rows are worked on by a kernel of their own, on the chunks of PagedAttentionExtension; their launches.
#include "flash_chunk.hpp"

namespace hipattn {

namespace flash {

// Launch index -> work item: workgroups go to the eight XCDs round-robin by launch index and
// each XCD has its own L2, so index i becomes item (i % 8) * (n / 8) + i / 8.  An XCD then walks
// a contiguous range of items ordered (batch, kv head, query tile descending, pair): the
// workgroups resident on it at one time share one K/V head, which stays in that L2, and the
// heaviest (latest) causal tiles of a head come first.  With an even number of query heads per
// kv head the two groups of a workgroup take two heads at the same query tile; otherwise they
// take two consecutive query tiles of one head.
template <bool kPad = false>
__device__ __forceinline__ Tile sdpa_group_tile(const SdpaParams& p, int group) {
    const int D = kPad ? p.head_dim : kD;
    const int G = small_div(p.num_heads_q, p.num_heads_kv);
    const int n_qt = (p.len_q + kTileQ - 1) / kTileQ;
    const bool pair_heads = (G & 1) == 0;
    const int slots = pair_heads ? n_qt : (n_qt + 1) / 2;  // query positions of a head's workgroups
    const int lanes = pair_heads ? G / 2 : G;              // workgroups per query position
    const int n_items = (int)gridDim.x;
    int item = (int)blockIdx.x;
    if ((n_items & 7) == 0) item = (item & 7) * (n_items >> 3) + (item >> 3);
    const int by_lane = small_div(item, lanes), li = item - by_lane * lanes;
    const int by_slot = small_div(by_lane, slots), slot = slots - 1 - (by_lane - by_slot * slots);
    const int b = small_div(by_slot, p.num_heads_kv), hkv = by_slot - b * p.num_heads_kv;
    const int h = hkv * G + (pair_heads ? 2 * li + group : li);
    const int qt = pair_heads ? slot : 2 * slot + group;
    Tile t;
    const int64_t qoff = (((int64_t)b * p.num_heads_q + h) * p.len_q + (int64_t)min(qt, n_qt - 1) * kTileQ) * D;
    t.q = (const uint16_t*)p.q + qoff;
    t.q_stride = D;
    t.out = (uint16_t*)p.out + qoff;
    t.out_stride = D;
    t.head_dim = D;
    t.rows = qt < n_qt ? min(kTileQ, p.len_q - qt * kTileQ) : 0;
    t.pos0 = qt * kTileQ;
    t.kv_len = p.len_kv;
    t.causal = p.causal;
    t.window = 0;
    t.q_dtype = p.dtype;
    t.out_dtype = p.dtype;
    const int64_t kvoff = ((int64_t)b * p.num_heads_kv + hkv) * p.len_kv * (D * 2);
    t.k = (const uint8_t*)p.k + kvoff;
    t.v = (const uint8_t*)p.v + kvoff;
    t.table = nullptr;
    t.table_len = 0;
    t.num_blocks = 0;
    t.block_stride = 0;
    t.block_size = 1;
    t.block_shift = 0;
    t.mask = nullptr;
    t.mask_row_bytes = 0;
    if (p.mask != nullptr) {
        const int64_t esz = p.mask_dtype == HIPATTN_U8 ? 1 : 2;
        t.mask = (const uint8_t*)p.mask +
                 ((int64_t)b * p.mask_stride[0] + (int64_t)h * p.mask_stride[1] + (int64_t)t.pos0 * p.mask_stride[2]) * esz;
        t.mask_row_bytes = p.mask_stride[2] * esz;
    }
    return t;
}

template <bool kBf16>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void sdpa_flash_kernel(SdpaParams p) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsBytes];
    const Tile t0 = sdpa_group_tile(p, 0), t1 = sdpa_group_tile(p, 1);
    run_both<kBf16, false, false>(t0, t1, lds, p.scale);
}

// The same for a head size between 64 and 128 (p.head_dim, a multiple of 8): the kPad form of the loop.
template <bool kBf16>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void sdpa_flash_padded_kernel(SdpaParams p) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsBytes];
    const Tile t0 = sdpa_group_tile<true>(p, 0), t1 = sdpa_group_tile<true>(p, 1);
    run_both<kBf16, false, false, 0, true>(t0, t1, lds, p.scale);
}

// The same with an attention mask (kMask 2: of the operands' type, added; 1: boolean bytes).
template <bool kBf16, int kMask>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void sdpa_flash_masked_kernel(SdpaParams p) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsBytes];
    const Tile t0 = sdpa_group_tile(p, 0), t1 = sdpa_group_tile(p, 1);
    run_both<kBf16, false, false, kMask>(t0, t1, lds, p.scale);
}

// ... and for a head size between 64 and 128.
template <bool kBf16, int kMask>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void sdpa_flash_masked_padded_kernel(SdpaParams p) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsBytes];
    const Tile t0 = sdpa_group_tile<true>(p, 0), t1 = sdpa_group_tile<true>(p, 1);
    run_both<kBf16, false, false, kMask, true>(t0, t1, lds, p.scale);
}

template <bool kBf16, bool kU8>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void paged_prefill_kernel(PagedParams p) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsBytes];
    paged_prefill_item<kBf16, kU8, false>(p, (int)blockIdx.x, lds);
}

// The same for a head size between 64 and 128 (16-bit caches): the kPad form of the loop.
template <bool kBf16>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void paged_prefill_padded_kernel(PagedParams p) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsBytes];
    paged_prefill_item<kBf16, false, true>(p, (int)blockIdx.x, lds);
}

}  // namespace flash

// Head size 128, and the smaller head sizes that are multiples of 8, which run the same kernel with rows of
// fewer columns in memory, 64 and 72 .. 96 and some calls of 104 .. 128 in sdpa_narrow.hip (16-byte aligned operands; the
// option sdpa_padded_rows = 0 leaves them to the plain kernels).  Measured on 4 x 2,048 tokens, 32 / 8 heads, causal: head size 64 0.079 ms there, 0.122 on
// padded rows, 0.153 in the plain head-64 kernel; head size 32 0.120 ms on padded rows.
bool sdpa_flash_supported(const SdpaParams& p) {
    if (!(p.dtype == HIPATTN_F16 || p.dtype == HIPATTN_BF16)) return false;
    if (p.head_dim != flash::kD) {
        const auto aligned16 = [](const void* q) { return ((uintptr_t)q & 15) == 0; };
        if (p.head_dim < 8 || p.head_dim > flash::kD || p.head_dim % 8 != 0 || !sdpa_padded_rows_enabled()) return false;
        if (!aligned16(p.q) || !aligned16(p.k) || !aligned16(p.v) || !aligned16(p.out)) return false;
    }
    // the kernel decodes its launch index with small_div: the number of workgroups must stay below 2^22
    const int64_t q_tiles = ((int64_t)p.len_q + flash::kTileQ - 1) / flash::kTileQ;
    return (int64_t)p.batch * p.num_heads_q * q_tiles < (int64_t(1) << 22);
}

// An attention mask the flash kernel takes: of the operands' type or boolean, its keys side by
// side, and every 16-byte piece the kernel loads aligned (the mask itself, and the steps from row
// to row, head to head and batch to batch; a step of 0 broadcasts).
bool sdpa_flash_mask_supported(const SdpaParams& p) {
    if (p.mask == nullptr || p.causal) return false;
    if (p.mask_dtype != p.dtype && p.mask_dtype != HIPATTN_U8) return false;
    if (p.mask_stride[3] != 1) return false;
    const int64_t per16 = p.mask_dtype == HIPATTN_U8 ? 16 : 8;
    if (((uintptr_t)p.mask & 15) != 0) return false;
    for (int i = 0; i < 3; i++)
        if (p.mask_stride[i] % per16 != 0) return false;
    return true;
}

hipError_t launch_sdpa_flash(const SdpaParams& p, hipStream_t stream, const KernelProbe& probe) {
    if (p.batch == 0 || p.len_q == 0) return hipSuccess;
    const int G = p.num_heads_q / p.num_heads_kv;
    const int n_qt = (p.len_q + flash::kTileQ - 1) / flash::kTileQ;
    const bool pair_heads = (G & 1) == 0;
    const int per_kv_head = pair_heads ? (G / 2) * n_qt : G * ((n_qt + 1) / 2);
    dim3 grid(per_kv_head * p.num_heads_kv * p.batch);
    if (probe.before) (void)hipEventRecord(probe.before, stream);
    const int mask = p.mask == nullptr ? 0 : (p.mask_dtype == HIPATTN_U8 ? 1 : 2);
    const dim3 block(flash::kThreads);
    if (p.head_dim != flash::kD) {  // (the kPad forms)
        if (p.dtype == HIPATTN_BF16) {
            if (mask == 0)
                hipLaunchKernelGGL(flash::sdpa_flash_padded_kernel<true>, grid, block, 0, stream, p);
            else if (mask == 2)
                hipLaunchKernelGGL((flash::sdpa_flash_masked_padded_kernel<true, 2>), grid, block, 0, stream, p);
            else
                hipLaunchKernelGGL((flash::sdpa_flash_masked_padded_kernel<true, 1>), grid, block, 0, stream, p);
        } else {
            if (mask == 0)
                hipLaunchKernelGGL(flash::sdpa_flash_padded_kernel<false>, grid, block, 0, stream, p);
            else if (mask == 2)
                hipLaunchKernelGGL((flash::sdpa_flash_masked_padded_kernel<false, 2>), grid, block, 0, stream, p);
            else
                hipLaunchKernelGGL((flash::sdpa_flash_masked_padded_kernel<false, 1>), grid, block, 0, stream, p);
        }
    } else if (p.dtype == HIPATTN_BF16) {
        if (mask == 0)
            hipLaunchKernelGGL(flash::sdpa_flash_kernel<true>, grid, block, 0, stream, p);
        else if (mask == 2)
            hipLaunchKernelGGL((flash::sdpa_flash_masked_kernel<true, 2>), grid, block, 0, stream, p);
        else
            hipLaunchKernelGGL((flash::sdpa_flash_masked_kernel<true, 1>), grid, block, 0, stream, p);
    } else {
        if (mask == 0)
            hipLaunchKernelGGL(flash::sdpa_flash_kernel<false>, grid, block, 0, stream, p);
        else if (mask == 2)
            hipLaunchKernelGGL((flash::sdpa_flash_masked_kernel<false, 2>), grid, block, 0, stream, p);
        else
            hipLaunchKernelGGL((flash::sdpa_flash_masked_kernel<false, 1>), grid, block, 0, stream, p);
    }
    hipError_t e = hipGetLastError();
    if (probe.after) (void)hipEventRecord(probe.after, stream);
    return e;
}

hipError_t launch_paged_prefill(const PagedParams& p, hipStream_t stream) {
    // the head sizes between 64 and 128 of a 16-bit cache: this kernel on rows of fewer columns
    const bool padded = p.head_dim > 64 && p.head_dim < flash::kD && p.head_dim % 8 == 0 && p.cache_dtype != HIPATTN_U8 &&
                        (((uintptr_t)p.q | (uintptr_t)p.key_cache | (uintptr_t)p.value_cache | (uintptr_t)p.out) & 15) == 0;
    // (ALiBi, attention sinks: the plain kernel has the distance term and the sink in its denominator; the tuned one
    // has no vector slot to spare for the one and was not given the other)
    if ((p.head_dim != flash::kD && !padded) || p.alibi_slopes || p.sinks) return launch_paged_prefill_small(p, stream);  // the plain kernel, padded columns
    const int G = p.num_heads_q / p.num_heads_kv;
    dim3 grid((unsigned)((int64_t)p.max_q_tiles * ((G & 1) == 0 ? p.num_heads_q / 2 : p.num_heads_q)));
    if (padded) {
        if (p.cache_dtype == HIPATTN_BF16)
            hipLaunchKernelGGL(flash::paged_prefill_padded_kernel<true>, grid, dim3(flash::kThreads), 0, stream, p);
        else
            hipLaunchKernelGGL(flash::paged_prefill_padded_kernel<false>, grid, dim3(flash::kThreads), 0, stream, p);
    } else if (p.cache_dtype == HIPATTN_BF16)
        hipLaunchKernelGGL((flash::paged_prefill_kernel<true, false>), grid, dim3(flash::kThreads), 0, stream, p);
    else if (p.cache_dtype == HIPATTN_U8)
        hipLaunchKernelGGL((flash::paged_prefill_kernel<false, true>), grid, dim3(flash::kThreads), 0, stream, p);
    else
        hipLaunchKernelGGL((flash::paged_prefill_kernel<false, false>), grid, dim3(flash::kThreads), 0, stream, p);
    return hipGetLastError();
}

}  // namespace hipattn
