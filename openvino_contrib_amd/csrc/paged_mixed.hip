// One launch for a mixed batch of PagedAttentionExtension: the rows of single-token sequences (the loop of
// paged_decode.hpp, bound by HBM) and the multi-token chunks (that of flash_chunk.hpp, bound by the matrix cores).
//
// Both take whole compute units.  The first workgroups, which are dispatched first, are the decode part's; the plan on
// the device has chosen how many of them work and the others leave at once, so that the chunks' workgroups find every
// compute unit the decode part does not keep.  (One sequence of a short context: no decode part, p.lone_tile.)  As two kernels, the chunks on a side stream, the fork and the join cost
// 20 to 27 us where there are no decode rows and about 10 where both parts are long.  Measured (us a step, two kernels -> one; 32 heads on 8 kv heads of 128):
// a prompt of 64 tokens 41 -> 14, of 1,000 58 -> 38, of 2,100 84 -> 67; 8 prompts of 1,000 142 -> 125, of 2,000 356 -> 339; two chunks of 200
// beside 20 decode rows 46 -> 37, beside 100 long ones 451 -> 444; 8 chunks of 512 beside 120 rows, 64 heads, 577 -> 567.
#include "flash_chunk.hpp"
#include "paged_decode.hpp"

namespace hipattn {

namespace {

template <bool kU8, bool kBf16, int kBlk, bool kPad>
__global__ __launch_bounds__(flash::kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void paged_mixed_kernel(PagedParams p, int decode_workgroups,
                                                                                                                int chunk_heads_kv) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[flash::kLdsBytes];
    if ((int)blockIdx.x < decode_workgroups) {
        const KvWriteParams none{};
        paged_decode_body<kU8, kBf16, 8, false, kD, kBlk, kPad>(p, none, 0, (int)blockIdx.x);
        return;
    }
    p.num_heads_kv = chunk_heads_kv;
    p.kv_share = 1;
    flash::paged_prefill_item<kBf16, kU8, kPad, kU8>(p, (int)blockIdx.x - decode_workgroups, lds);
}

template <bool kU8, bool kBf16, bool kPad>
void launch_blk(const PagedParams& p, int decode_workgroups, int chunk_heads_kv, dim3 grid, hipStream_t stream) {
    const dim3 block(flash::kThreads);
    if (p.block_size == 32)
        hipLaunchKernelGGL((paged_mixed_kernel<kU8, kBf16, 32, kPad>), grid, block, 0, stream, p, decode_workgroups, chunk_heads_kv);
    else if (p.block_size == 16)
        hipLaunchKernelGGL((paged_mixed_kernel<kU8, kBf16, 16, kPad>), grid, block, 0, stream, p, decode_workgroups, chunk_heads_kv);
    else
        hipLaunchKernelGGL((paged_mixed_kernel<kU8, kBf16, 0, kPad>), grid, block, 0, stream, p, decode_workgroups, chunk_heads_kv);
}

}  // namespace

// Head size 128, and 16-bit caches of the sizes between 64 and 128 on aligned rows: what both loops are built for.  (The sinks
// of a chunk are known to the kernel of flash_small.hip only.)
bool paged_mixed_supported(const PagedParams& p) {
    if (p.sinks || p.alibi_slopes) return false;
    if (p.head_dim == kD) return true;
    return p.cache_dtype != HIPATTN_U8 && (((uintptr_t)p.q | (uintptr_t)p.key_cache | (uintptr_t)p.value_cache | (uintptr_t)p.out) & 15) == 0;
}

hipError_t launch_paged_mixed(const PagedParams& p, int chunk_heads_kv, hipStream_t stream) {
    // (workgroups go to the XCDs round-robin and the chunks' order counts on that: a multiple of eight in front of them)
    const int decode_workgroups = p.lone_tile ? 0 : (p.num_waves / 8 + 7) / 8 * 8;
    const int G = p.num_heads_q / chunk_heads_kv;
    const dim3 grid((unsigned)(decode_workgroups + (int64_t)p.max_q_tiles * ((G & 1) == 0 ? p.num_heads_q / 2 : p.num_heads_q)));
    const bool bf16 = p.cache_dtype == HIPATTN_BF16;
    if (p.cache_dtype == HIPATTN_U8)
        launch_blk<true, false, false>(p, decode_workgroups, chunk_heads_kv, grid, stream);
    else if (p.head_dim == kD)
        bf16 ? launch_blk<false, true, false>(p, decode_workgroups, chunk_heads_kv, grid, stream)
             : launch_blk<false, false, false>(p, decode_workgroups, chunk_heads_kv, grid, stream);
    else
        bf16 ? launch_blk<false, true, true>(p, decode_workgroups, chunk_heads_kv, grid, stream)
             : launch_blk<false, false, true>(p, decode_workgroups, chunk_heads_kv, grid, stream);
    return hipGetLastError();
}

}  // namespace hipattn
