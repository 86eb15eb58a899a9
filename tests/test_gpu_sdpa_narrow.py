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


def biased_rows(Lq, Lk, dtype):
    """(mask, the same with a constant taken off every row), row after row another kind: a constant, one of two constants on
    either half of the keys, very low keys before and behind a constant, a falling and a rising ramp."""
    constants, mask = np.zeros((Lq, 1), np.float32), np.zeros((Lq, Lk), np.float32)
    fp16 = dtype == W.F16
    step = 2 if fp16 else 16  # (the type's spacing there)
    near = [-2800 - step * i for i in range(27 if fp16 else 8)]
    far = [-100.0, -700.0, 96.0, 3072.0, -12288.0] + ([-65504.0, 61440.0] if fp16 else [-131072.0, 2.0 ** 40])
    lowest = -65504.0 if fp16 else -(2.0 ** 100)
    half = np.arange(Lk) < Lk // 2
    kinds = [(c, 0.0 * half) for c in near + far]
    kinds += [(c, np.where(half if flip else ~half, -float(step), 0.0)) for c in near for flip in (False, True)]
    kinds += [(c, np.where(half if flip else ~half, -np.inf, 0.0)) for c in near + far[:4] for flip in (False, True)]
    ramp = np.arange(Lk) * -float(step)
    kinds += [(c, r) for c in near + far[:2] for r in (ramp, ramp[::-1])]
    for i in range(Lq):
        c, d = kinds[(i * 7) % len(kinds)]
        constants[i], mask[i] = c, np.where(np.isneginf(d), lowest, c + d)
    mask = W.to_storage(mask, dtype)[1]
    return mask, mask - constants


# (in the order of the wavefronts that share 32 query rows: one, two, four)
@pytest.mark.parametrize("dtype", [W.F16, W.BF16])
@pytest.mark.parametrize("shape", [(4, 64, 8, 130, 400, 64), (2, 64, 8, 130, 400, 96), (2, 64, 8, 130, 250, 128), (2, 24, 24, 300, 300, 64), (2, 24, 6, 300, 300, 96),
                                   (2, 16, 16, 300, 300, 128), (1, 4, 2, 130, 1000, 64), (1, 16, 16, 300, 300, 96), (1, 8, 8, 300, 300, 104)])
def test_a_constant_added_to_a_row_changes_nothing(hip, oracle, dtype, shape):
    """The softmax is the same whatever is added to all scores of a row.  The constants are values of the type, so that the
    oracle's mask without them is exact, and what the kernel takes off mask * log2(e) is the same for all keys of the row."""
    B, Hq, Hkv, Lq, Lk, D = shape
    case = W.make_sdpa_case(24, B, Hq, Hkv, Lq, Lk, D, dtype)
    m, shifted = biased_rows(Lq, Lk, dtype)
    out, _ = H.run_sdpa_masked(hip, case, m, mask_dtype=dtype)
    ref = oracle.sdpa_masked(case["q"], case["k"], case["v"], shifted)
    assert H.scaled_bound_error(out, ref, "row constants") <= (2e-3 if dtype == W.F16 else 1e-2)
