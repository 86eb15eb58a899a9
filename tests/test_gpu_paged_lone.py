"""A paged call of one sequence whose lengths only the device knows: a single token behind the flag for any lengths, a single token among
padding, and a recorded call replayed with other lengths.  Whatever the sequence turns out to hold, its rows are attended (against the
oracle, into an output filled before), and padding tokens get none."""
import ctypes

import numpy as np
import pytest

from openvino_contrib_amd import workloads as W
import helpers as H
from test_gpu_graph import CAPTURE_MODE_RELAXED, hip_runtime

pytestmark = pytest.mark.gpu

# the kernel of both parts: head size 128 with any cache, 72 .. 120 with 16-bit caches
SHAPES = [(W.F16, 32, 128, (8, 2)), (W.BF16, 16, 128, (4, 1)), (W.U8, 32, 128, (8, 2)), (W.U8, 16, 128, (3, 3)), (W.F16, 64, 128, (3, 1)),
          (W.F16, 32, 96, (4, 2)), (W.BF16, 16, 72, (2, 2)), (W.F16, 32, 128, (48, 1))]
TOLERANCE = {W.F16: 2e-3, W.U8: 1e-2, W.BF16: 2e-2}  # as in test_gpu_paged_mixed.py: the operands' types


def paged_case(seed, past, new, cache, block, size, heads, tokens=None, first=0):
    """One sequence of `new` tokens, token `first` of `tokens`; the others are padding."""
    q = W.BF16 if cache == W.BF16 else W.F16
    case = W.make_paged_case(seed, [(past, tokens or new)], heads[0], heads[1], size, block, q, q, cache)
    case["subsequence_begins"] = np.array([first, first + new], np.int32)
    case["max_context_len"] = past + new
    return case


def check(hip, oracle, case, flags=0, max_context_len=None):
    # (the oracle walks the sequence's own tokens: rows of padding stay what its output holds)
    ref, okc, ovc = H.oracle_paged(oracle, case)
    dev = H.PagedDeviceCase(hip, case)
    out, path = dev.run(flags, max_context_len=max_context_len)
    kc, vc = dev.caches()
    dev.free()
    assert path == "paged_mfma"
    b0, b1 = case["subsequence_begins"]
    assert H.scaled_bound_error(out[b0:b1], ref[b0:b1], "tokens %d..%d" % (b0, b1)) <= TOLERANCE[case["cache_dtype"]]
    np.testing.assert_array_equal(kc, okc)
    np.testing.assert_array_equal(vc, ovc)
    return out


@pytest.mark.parametrize("past", [0, 5, 300, 2500])
@pytest.mark.parametrize("cache,block,size,heads", SHAPES)
def test_one_token_of_one_sequence(hip, oracle, cache, block, size, heads, past):
    for flags in (0, hip.PA_ANY_LENGTHS):
        check(hip, oracle, paged_case(31, past, 1, cache, block, size, heads), flags)


@pytest.mark.parametrize("past,new,first,tokens", [(300, 1, 0, 8), (300, 1, 2, 8), (2500, 1, 7, 8), (0, 1, 1, 2), (40, 5, 2, 8), (300, 0, 3, 8), (6000, 1, 3, 500), (0, 400, 3, 500)])
@pytest.mark.parametrize("cache,block,size,heads", SHAPES)
def test_one_sequence_among_padding_tokens(hip, oracle, cache, block, size, heads, past, new, first, tokens):
    case = paged_case(32, past, new, cache, block, size, heads, tokens, first)
    for bound in (None, 0):  # (0: the caller knows no bound on the context)
        check(hip, oracle, case, max_context_len=bound)


@pytest.mark.parametrize("cache,block,size,heads", SHAPES)
def test_one_token_without_a_block_table_is_zeros(hip, oracle, cache, block, size, heads):
    case = paged_case(33, 20, 1, cache, block, size, heads, 8, 2)
    case["block_indices_begins"] = np.array([0, 0], np.int32)
    out = check(hip, oracle, case)
    assert not out[2].any()


@pytest.mark.parametrize("cache,block,size,heads", SHAPES[:4] + SHAPES[5:6])
def test_a_recorded_call_of_one_sequence_takes_any_lengths(hip, oracle, cache, block, size, heads):
    recorded = paged_case(34, 90, 8, cache, block, size, heads)
    rt = hip_runtime()
    stream = hip.Stream()
    dev = H.PagedDeviceCase(hip, paged_case(34, 3000, 8, cache, block, size, heads))
    begins, past = (hip.DeviceBuffer.from_numpy(recorded[n]) for n in ("subsequence_begins", "past_lens"))
    desc = H.pa_desc(hip, dict(dev.case, max_context_len=98))
    ws = hip.DeviceBuffer(hip.paged_attention_workspace_size(desc))

    def call(d):
        hip.paged_attention(d, dev.q, dev.k_new, dev.v_new, dev.key_cache, dev.value_cache, past, begins, dev.block_indices,
                            dev.block_indices_begins, dev.out, ws, stream)

    call(H.pa_desc(hip, dict(dev.case, max_context_len=98), flags=hip.PA_SKIP_CACHE_WRITE))  # eager: whatever a device's first call sets up
    graph, graph_exec = ctypes.c_void_p(), ctypes.c_void_p()
    assert rt.hipStreamBeginCapture(stream.handle, CAPTURE_MODE_RELAXED) == 0
    try:
        call(desc)
    finally:
        status = rt.hipStreamEndCapture(stream.handle, ctypes.byref(graph))
    assert status == 0 and graph.value
    assert rt.hipGraphInstantiate(ctypes.byref(graph_exec), graph, None, None, 0) == 0
    try:
        for length, new, first in ((90, 8, 0), (700, 1, 0), (2999, 5, 2), (3000, 1, 4), (0, 1, 7)):
            case = dict(dev.case, past_lens=np.array([length], np.int32), subsequence_begins=np.array([first, first + new], np.int32))
            case["key_cache"], case["value_cache"] = dev.caches()
            ref, okc, ovc = H.oracle_paged(oracle, case)
            begins.upload(case["subsequence_begins"], stream)
            past.upload(case["past_lens"], stream)
            dev.out.fill(0xFF, stream)
            assert rt.hipGraphLaunch(graph_exec, stream.handle) == 0
            got = H.storage_to_f32(dev.out.download(np.uint16, (case["T"], case["Hq"] * case["D"]), stream), case["q_dtype"])
            rows = slice(first, first + new)
            assert H.scaled_bound_error(got[rows], ref[rows], "replay %d %d" % (length, new)) <= TOLERANCE[cache]
            kc, vc = dev.caches()
            np.testing.assert_array_equal(kc, okc)
            np.testing.assert_array_equal(vc, ovc)
    finally:
        rt.hipGraphExecDestroy(graph_exec)
        rt.hipGraphDestroy(graph)
        for b in (ws, begins, past):
            b.free()
        dev.free()
        stream.close()
