"""Dense attention at head sizes 64 and 72 .. 128: edges of the 32-row and 64-key tiles, rows that leave wavefronts of a
workgroup idle, key halves that are masked as a whole, and masks whose rows start at any address, against the oracle.
Bounds: the repository's 2e-3 (fp16) and 1e-2 (bf16) on outputs within [-4, 4] (scaled where they leave [-1, 1])."""
import numpy as np
import pytest

import helpers as H
from openvino_contrib_amd import workloads as W

pytestmark = pytest.mark.gpu

# (batch, heads, kv heads, queries, keys, head size)
SHAPES = [(1, 1, 1, 1, 1, 64), (1, 2, 1, 33, 31, 64), (2, 4, 2, 32, 33, 64), (1, 3, 3, 129, 65, 64), (1, 8, 8, 97, 95, 64),
          (3, 2, 2, 161, 577, 64), (1, 2, 1, 300, 129, 64), (1, 1, 1, 128, 128, 96), (2, 3, 1, 50, 97, 96), (1, 4, 4, 65, 191, 72),
          (1, 2, 2, 31, 64, 80), (2, 6, 3, 200, 321, 80), (1, 2, 1, 130, 63, 88), (1, 4, 2, 33, 31, 128), (1, 2, 2, 129, 321, 128), (2, 3, 3, 64, 97, 104),
          (3, 4, 1, 161, 129, 120)]


@pytest.mark.parametrize("dtype", [W.F16, W.BF16])
@pytest.mark.parametrize("mask", ["none", "causal", "padding", "scattered", "bias"])
@pytest.mark.parametrize("shape", SHAPES)
def test_sdpa_narrow(hip, oracle, shape, mask, dtype):
    B, Hq, Hkv, Lq, Lk, D = shape
    case = W.make_sdpa_case(21, B, Hq, Hkv, Lq, Lk, D, dtype)
    rng = np.random.default_rng(4)
    if mask in ("none", "causal"):
        out, _ = H.run_sdpa(hip, case, mask == "causal")
        ref = oracle.sdpa(case["q"], case["k"], case["v"], causal=mask == "causal")
    else:
        if mask == "padding":
            m = np.arange(Lk)[None, None, None, :] < rng.integers(0, Lk + 1, (B, 1, 1, 1))  # (a row of zero keys gives zeros)
        elif mask == "scattered":
            m = rng.random((1, Hq, Lq, Lk)) < 0.3
        else:
            m = W.to_storage(rng.standard_normal((B, 1, Lq, Lk)).astype(np.float32), dtype)[1]
            m[..., Lk - Lk // 3:] = -np.inf
        out, _ = H.run_sdpa_masked(hip, case, m, mask_dtype=dtype)
        ref = oracle.sdpa_masked(case["q"], case["k"], case["v"], m)
    assert np.isfinite(out).all()
    assert H.scaled_bound_error(out, ref, "narrow heads") <= (2e-3 if dtype == W.F16 else 1e-2)


@pytest.mark.parametrize("dtype", [W.F16, W.BF16])
def test_growing_scores(hip, oracle, dtype):
    """Scores that outgrow every reference taken before them: the accumulators and the scores already computed move along."""
    case = W.make_sdpa_case(22, 1, 2, 2, 70, 400, 64, dtype)
    case["k"][..., 0] = np.linspace(-200, 200, 400)
    case["q"][..., 0] = 1.0
    for n in "qk":
        case[n + "_store"], case[n] = W.to_storage(case[n], dtype)
    out, _ = H.run_sdpa(hip, case, False)
    # the products' operands: q * scale * log2(e) is rounded to 16 bits, 2^-11 (2^-8) of scores up to 25 nats
    ref = oracle.sdpa(case["q"], case["k"], case["v"])
    assert np.isfinite(out).all()
    assert H.max_abs(out, ref) <= (0.05 if dtype == W.F16 else 0.4)


@pytest.mark.parametrize("dtype", [W.F16, W.BF16])
@pytest.mark.parametrize("shape", [(2, 4, 2, 70, 300, 64), (1, 2, 2, 33, 90, 96), (1, 24, 24, 640, 200, 64), (1, 2, 1, 140, 500, 128)])
def test_masks_of_the_lowest_value(hip, oracle, dtype, shape):
    """Keys masked by the type's lowest value (fp16: finite after the change of base), the first ones of every row, some rows as
    a whole: the kept keys weigh as if the others were not there, and a row of none but such keys is their mean weighted by
    scores that the mask has rounded away (bf16: -inf after the change of base, and zeros)."""
    B, Hq, Hkv, Lq, Lk, D = shape
    case = W.make_sdpa_case(23, B, Hq, Hkv, Lq, Lk, D, dtype)
    lowest = -65504.0 if dtype == W.F16 else float(np.frombuffer(np.uint32(0xff7f0000).tobytes(), np.float32)[0])
    m = np.zeros((1, 1, Lq, Lk), np.float32)
    m[..., :75] = lowest
    m[:, :, Lq // 2:Lq // 2 + 3] = lowest
    gone = m == lowest
    case["k"][:, :, :75] *= 0.0  # (equal scores: the mean of a row of such keys is exact whatever their rounding)
    case["k"][..., 0] = 0
    case["q"][:, :, Lq // 2:Lq // 2 + 3] = 0
    for n in "qk":
        case[n + "_store"], case[n] = W.to_storage(case[n], dtype)
    out, _ = H.run_sdpa_masked(hip, case, m, mask_dtype=dtype)
    ref = oracle.sdpa_masked(case["q"], case["k"], case["v"], np.where(gone, -np.inf, 0).astype(np.float32))
    rows = slice(Lq // 2, Lq // 2 + 3)
    if dtype == W.F16:
        ref[:, :, rows] = np.repeat(case["v"].mean(2, keepdims=True), Hq // Hkv, axis=1)
    else:
        ref[:, :, rows] = 0
    assert H.scaled_bound_error(out, ref, "lowest mask") <= (2e-3 if dtype == W.F16 else 1e-2)
