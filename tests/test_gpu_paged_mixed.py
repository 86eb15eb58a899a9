"""Mixed batches in one launch (paged_mixed.hip): every cache type and block size the kernel is built for, on batches at
the edges of its grid -- one sequence (no decode part), chunks only, decode rows beside one short chunk, empty sequences,
query heads that do not pair -- against the oracle and against one kernel after the other."""
import numpy as np
import pytest

from openvino_contrib_amd import capi
from openvino_contrib_amd import workloads as W
import helpers as H

pytestmark = pytest.mark.gpu

BATCHES = {
    "one_chunk": [(0, 65)],
    "one_chunk_with_past": [(300, 129)],
    "chunks_only": [(0, 2), (17, 128), (64, 130)],
    "short_chunk_many_rows": [(0, 2)] + [(37 * i, 1) for i in range(1, 30)],
    "empty_sequences": [(0, 0), (900, 1), (0, 0), (100, 200), (5, 1), (0, 0)],
}


@pytest.mark.parametrize("batch", sorted(BATCHES))
@pytest.mark.parametrize("cache,block,size,heads", [(W.F16, 32, 128, (8, 2)), (W.BF16, 16, 128, (8, 2)), (W.U8, 32, 128, (8, 2)), (W.U8, 16, 128, (3, 3)),
                                                    (W.F16, 64, 128, (3, 1)), (W.U8, 128, 128, (8, 1)), (W.BF16, 32, 96, (4, 2)), (W.F16, 16, 72, (2, 2)),
                                                    (W.F16, 64, 104, (8, 2)), (W.F16, 32, 128, (48, 1))])
def test_mixed_batches_in_one_launch(hip, oracle, batch, cache, block, size, heads):
    q = W.BF16 if cache == W.BF16 else W.F16
    case = W.make_paged_case(71, BATCHES[batch], heads[0], heads[1], size, block, q, q, cache)
    ref = H.oracle_paged(oracle, case)[0]
    dev = H.PagedDeviceCase(hip, case)
    out, path = dev.run()
    again, _ = dev.run()
    dev.free()
    assert path == "paged_mfma"
    np.testing.assert_array_equal(out, again)
    # fp16 operands 2e-3, u8 rows dequantised to fp16 1e-2; bf16 probabilities and scaled queries (2^-9 each) reach 1.2e-2 in
    # chunk rows on such data
    tol = {W.F16: 2e-3, W.U8: 1e-2, W.BF16: 2e-2}[cache]
    assert H.scaled_bound_error(out, ref, "%s cache %d" % (batch, cache)) <= tol
    capi.check(capi.lib().hipattn_set_option(b"mixed_overlap", 0))
    try:
        serial = H.PagedDeviceCase(hip, case)
        alone, _ = serial.run()
        serial.free()
    finally:
        capi.check(capi.lib().hipattn_set_option(b"mixed_overlap", -1))
    assert H.scaled_bound_error(out, alone, "against one kernel after the other") <= tol


@pytest.mark.parametrize("block,heads", [(32, (8, 2)), (16, (3, 3)), (128, (8, 8)), (32, (48, 1))])
@pytest.mark.parametrize("seqs", [[(0, 384)], [(0, 33), (0, 1), (0, 417), (5, 400), (0, 0), (0, 383), (200, 1), (0, 640)], [(0, 511), (64, 2), (0, 385), (0, 0), (0, 700)]])
def test_new_prompts_read_the_rows_that_the_writer_quantised(hip, oracle, seqs, block, heads):
    """u8 caches: sequences of 384 new tokens or more without cached ones take their rows from the writer's dequantised copy, others from the cache, in one call: the
    chunk rows bit for bit those of the kernel that dequantises the cache's rows itself, with whole and missing table entries
    (the first block of a sequence among them)."""
    case = W.make_paged_case(5, seqs, heads[0], heads[1], 128, block, W.BF16, W.BF16, W.U8)
    for broken in (False, True):
        if broken:  # every fifth entry names no block
            case["block_indices"] = case["block_indices"].copy()
            case["block_indices"][::5] = -7
        ref = H.oracle_paged(oracle, case)[0]
        results = []
        for overlap in (-1, 0):
            capi.check(capi.lib().hipattn_set_option(b"mixed_overlap", overlap))
            try:
                dev = H.PagedDeviceCase(hip, case)
                results.append(dev.run()[0])
                dev.free()
            finally:
                capi.check(capi.lib().hipattn_set_option(b"mixed_overlap", -1))
        begins = case["subsequence_begins"]
        chunk = np.concatenate([np.arange(begins[s], begins[s + 1]) for s in range(len(seqs)) if seqs[s][1] > 1])
        np.testing.assert_array_equal(results[0][chunk], results[1][chunk])
        assert H.scaled_bound_error(results[0], ref, "%s broken %d" % (seqs, broken)) <= 1e-2


@pytest.mark.parametrize("room", [0, 1])
def test_new_prompts_without_room_for_the_copy(hip, oracle, room):
    """A caller with the workspace of a call without such prompts, or a byte less than the copy takes: the rows come from the cache, bit for bit the same."""
    seqs = [(0, 640), (0, 33), (200, 1), (0, 417)]
    case = W.make_paged_case(6, seqs, 8, 2, 128, 32, W.BF16, W.BF16, W.U8)
    dev = H.PagedDeviceCase(hip, case)
    with_copy = dev.run()[0]
    desc = H.pa_desc(hip, case)
    whole, without = hip.paged_attention_workspace_size(desc), hip.paged_attention_workspace_size(H.pa_desc(hip, case, max_context_len=100))
    assert without < whole
    ws = hip.DeviceBuffer(whole - 1 if room else without)
    dev.out.fill(0xFF)
    hip.paged_attention(desc, dev.q, dev.k_new, dev.v_new, dev.key_cache, dev.value_cache, dev.past_lens, dev.subsequence_begins, dev.block_indices,
                        dev.block_indices_begins, dev.out, ws)
    out = H.storage_to_f32(dev.out.download(np.uint16, with_copy.shape), W.BF16)
    np.testing.assert_array_equal(out, with_copy)
    assert H.scaled_bound_error(out, H.oracle_paged(oracle, case)[0], "no room") <= 1e-2
    ws.free()
    dev.free()
