"""Decode steps of few sequences: the number of wavefronts the plan lets work, and the merge of many pieces per
(sequence, kv head) by several wavefronts.  Against the oracle, at the bounds of the decode tests (max-abs 2e-3
for fp16 operands, 1e-2 for u8 and bf16 caches; outputs of N(0,1) values averaged over a context stay within [-4, 4])."""
import pytest

import helpers as H
from openvino_contrib_amd import workloads as W

pytestmark = pytest.mark.gpu

# contexts: a single token; both sides of one 32-token unit and of a piece; as many units as wavefronts with and
# without the switch cost; 64 and more pieces per segment; uneven sequences beside each other; more than 128 segments
BATCHES = [[1], [32], [33], [255, 1], [778], [5000], [16384], [256, 4096, 33, 1700], [20] * 40, [3000] * 17]


@pytest.mark.parametrize("cache", [W.F16, W.BF16, W.U8])
@pytest.mark.parametrize("contexts", BATCHES, ids=lambda c: "x".join(map(str, c[:2])) + "_%d" % len(c))
@pytest.mark.parametrize("heads,D,block", [((32, 8), 128, 32), ((8, 8), 64, 16), ((4, 2), 256, 32)])
def test_decode_of_few_sequences(hip, oracle, contexts, cache, heads, D, block):
    if D == 256 and len(contexts) > 4:
        pytest.skip("the large batches at the head sizes of the other kernels only")
    q = W.BF16 if cache == W.BF16 else W.F16
    case = W.make_paged_case(11, [(c - 1, 1) for c in contexts], heads[0], heads[1], D, block, q, q, cache)
    dev = H.PagedDeviceCase(hip, case, out_dtype=W.F32)
    out, path = dev.run()
    ref, kc, vc = H.oracle_paged(oracle, case)
    got_kc, got_vc = dev.caches()
    dev.free()
    assert path == "paged_mfma"
    assert (got_kc == kc).all() and (got_vc == vc).all()
    assert H.scaled_bound_error(out, ref, "decode of few") <= (2e-3 if cache == W.F16 else 1e-2)


# either side of the lines the schedule draws: four blocks and five (and eight, beside a chunk); 120 and 128 segments; three pieces
# to a segment and more; eight pieces and more in the merge; a wavefront count that is rounded
LINES = [[(127, 1)] * 5, [(128, 1)] * 5, [(100, 1)] * 15, [(100, 1)] * 16, [(299, 1)] * 15, [(299, 1)] * 16, [(299, 1)] * 49, [(859, 1)] * 16,
         [(30, 1), (2000, 1)] * 9, [(0, 60)], [(0, 250), (99, 1)], [(0, 257), (299, 1)], [(3, 40), (3999, 1), (100, 1)]]


@pytest.mark.parametrize("window", [0, 100])
@pytest.mark.parametrize("cache", [W.F16, W.U8])
@pytest.mark.parametrize("seqs", LINES, ids=lambda s: "%dx%d_%d" % (len(s), s[-1][0], s[-1][1]))
def test_lines_of_the_schedule(hip, oracle, seqs, cache, window):
    """The bound on the contexts that the caller gives decides where pieces meet; any bound that holds gives the same rows."""
    case = W.make_paged_case(12, seqs, 32, 8, 128, 32, W.F16, W.F16, cache, sliding_window=window)
    ref, _, _ = H.oracle_paged(oracle, case)
    for bound in (case["max_context_len"], 1 << 20):
        dev = H.PagedDeviceCase(hip, case, out_dtype=W.F32)
        out, path = dev.run(max_context_len=bound)
        dev.free()
        assert path == "paged_mfma"
        assert H.scaled_bound_error(out, ref, "lines") <= (2e-3 if cache == W.F16 else 1e-2)
