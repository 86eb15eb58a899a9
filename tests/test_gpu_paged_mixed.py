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
