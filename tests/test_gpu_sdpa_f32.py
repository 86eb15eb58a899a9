"""fp32 attention on the fp32 matrix cores: the edges of its row and key tiles, of the split of the keys over
wavefronts and of the head sizes, against the oracle.  Bound: 1e-4, the repository's for fp32 operands; sums of
len_kv fp32 terms of size 1 differ from the oracle's by less than len_kv * 6e-8 of their value."""
import numpy as np
import pytest

import helpers as H
from openvino_contrib_amd import workloads as W

pytestmark = pytest.mark.gpu

# (batch, heads, kv heads, queries, keys, head size): one row and one key; tiles of 16 and 32 rows and keys and one
# more; keys that leave some of the wavefronts without any; rows enough for two row tiles per wavefront; head
# sizes at and beside the two the kernel is built for
SHAPES = [(1, 1, 1, 1, 1, 64), (1, 2, 1, 17, 15, 64), (2, 4, 2, 16, 33, 64), (1, 8, 8, 128, 128, 64), (1, 3, 3, 31, 129, 128),
          (3, 2, 2, 65, 64, 96), (1, 4, 1, 33, 47, 4), (2, 2, 2, 50, 17, 68), (4, 16, 16, 161, 95, 64), (3, 16, 4, 257, 260, 128),
          (16, 16, 16, 97, 40, 32), (1, 1, 1, 5, 700, 128), (2, 12, 12, 384, 384, 64)]


@pytest.mark.parametrize("mask", ["none", "causal", "padding", "float", "f16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_sdpa_f32(hip, oracle, shape, mask):
    B, Hq, Hkv, Lq, Lk, D = shape
    case = W.make_sdpa_case(7, B, Hq, Hkv, Lq, Lk, D, W.F32)
    rng = np.random.default_rng(3)
    m = None
    if mask == "padding":
        m = np.arange(Lk)[None, None, None, :] < rng.integers(0, Lk + 1, (B, 1, 1, 1))  # (a row of zero keys gives zeros)
    elif mask in ("float", "f16"):
        m = rng.standard_normal((1, Hq, Lq, Lk)).astype(np.float32)
        m[..., Lk - Lk // 3:] = -np.inf
    if m is None:
        out, _ = H.run_sdpa(hip, case, mask == "causal")
        ref = oracle.sdpa(case["q"], case["k"], case["v"], causal=mask == "causal")
    else:
        out, _ = H.run_sdpa_masked(hip, case, m.astype(np.float16) if mask == "f16" else m)
        ref = oracle.sdpa_masked(case["q"], case["k"], case["v"], m.astype(np.float16).astype(np.float32) if mask == "f16" else m)
    assert np.isfinite(out).all()
    assert H.max_abs(out, ref) <= 1e-4


@pytest.mark.parametrize("shape", [(2, 4, 2, 33, 47, 64), (1, 2, 2, 20, 70, 96), (1, 4, 4, 160, 200, 128)])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_masked_keys_may_hold_anything(hip, oracle, shape, value):
    """Value rows of keys that a row does not attend, infinite or NaN: the row is what it is without them."""
    B, Hq, Hkv, Lq, Lk, D = shape
    case = W.make_sdpa_case(8, B, Hq, Hkv, Lq, Lk, D, W.F32)
    cut = Lk - 5
    m = np.broadcast_to(np.arange(Lk) < cut, (1, 1, 1, Lk)).copy()
    ref = oracle.sdpa_masked(case["q"], case["k"], case["v"], m)
    case["v"][:, :, cut:, 0] = value
    for form in (m, np.where(m, 0.0, -np.inf).astype(np.float32)):
        out, _ = H.run_sdpa_masked(hip, case, form)
        assert H.max_abs(out, ref) <= 1e-4
    case = W.make_sdpa_case(9, B, Hq, Hkv, Lq, Lk, D, W.F32)
    ref = oracle.sdpa(case["q"], case["k"], case["v"], causal=True)
    at = Lq // 2
    case["v"][:, :, at, :] = value  # rows from `at` on attend it
    out, _ = H.run_sdpa(hip, case, True)
    assert H.max_abs(out[:, :, :at], ref[:, :, :at]) <= 1e-4
    assert not np.isfinite(out[:, :, at:]).any()


def test_large_values_beside_growing_scores(hip, oracle):
    """Scores that grow by some 2^20 along the keys and values near the largest fp32: the sums stay finite."""
    case = W.make_sdpa_case(10, 1, 2, 2, 40, 300, 64, W.F32)
    case["q"][..., 0] = 1.0
    case["k"][..., 0] = np.linspace(0, 160, 300, dtype=np.float32)  # (times 1 / sqrt(64))
    case["v"] *= np.float32(2e37)
    out, _ = H.run_sdpa(hip, case, False)
    ref = oracle.sdpa(case["q"], case["k"], (case["v"] / np.float32(2e37)))
    assert np.isfinite(out).all()
    assert H.max_abs(out / np.float32(2e37), ref) <= 1e-4


@pytest.mark.parametrize("mask_dtype", [W.F32, W.F16])
@pytest.mark.parametrize("shape", [(1, 2, 1, 33, 64, 64), (2, 2, 2, 20, 200, 128), (1, 4, 4, 160, 47, 32)])
def test_nan_masks_reach_their_rows(hip, oracle, shape, mask_dtype):
    """Sixteen keys whose mask is NaN for every row of a tile, beside -inf and beside finite values: the rows are NaN, as
    rows with one such key are; the rows of a tile without any are what they are."""
    B, Hq, Hkv, Lq, Lk, D = shape
    case = W.make_sdpa_case(11, B, Hq, Hkv, Lq, Lk, D, W.F32)
    m = np.zeros((1, 1, Lq, Lk), np.float32)
    m[..., 16:32] = np.nan
    m[..., 32:] = -np.inf
    out, _ = H.run_sdpa_masked(hip, case, m, mask_dtype=mask_dtype)
    assert np.isnan(out).all()
    m[..., 16:32] = -np.inf
    m[:, :, 3, 18] = np.nan
    out, _ = H.run_sdpa_masked(hip, case, m, mask_dtype=mask_dtype)
    assert np.isnan(out[:, :, 3]).all()
    m[:, :, 3, 18] = -np.inf
    ref = oracle.sdpa_masked(case["q"], case["k"], case["v"], m)
    rest = np.arange(Lq) != 3
    assert H.max_abs(out[:, :, rest], ref[:, :, rest]) <= 1e-4


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_an_infinite_value_stays_in_its_column(hip, oracle, shape, masked):
    """Every row attends a key with one infinite value: its column is infinite, the others are what they are.  Such rows are
    worked again, one after the other."""
    B, Hq, Hkv, Lq, Lk, D = shape
    case = W.make_sdpa_case(12, B, Hq, Hkv, Lq, Lk, D, W.F32)
    m = np.zeros((1, 1, Lq, Lk), np.float32)
    m[..., Lk // 2 + 1:] = -np.inf
    ref = oracle.sdpa_masked(case["q"], case["k"], case["v"], m) if masked else oracle.sdpa(case["q"], case["k"], case["v"])
    case["v"][:, :, Lk // 2, D - 1] = np.inf
    out, _ = H.run_sdpa_masked(hip, case, m) if masked else H.run_sdpa(hip, case, False)
    assert np.isposinf(out[..., D - 1]).all()
    assert H.max_abs(out[..., :D - 1], ref[..., :D - 1]) <= 1e-4
