"""Dense 16-bit attention in each kernel that takes it, whichever the rule of choice picks: the shapes, growing scores and masks
of the general tests in the tuned head-128 kernel (option sdpa_narrow 0) and in the one of small workgroups (2), there with
one, two and four wavefronts to 32 query rows.  Bounds: those of the tests that are run again."""
import numpy as np
import pytest

import helpers as H
import test_gpu_parity as parity
import test_gpu_random as random_tests
import test_gpu_sdpa_narrow as narrow
from openvino_contrib_amd import workloads as W

pytestmark = pytest.mark.gpu

TOL = {W.F16: 2e-3, W.BF16: 1e-2}


def parameters(test, names):
    """The values that a test is parametrised with."""
    return next(m.args[1] for m in test.pytestmark if m.name == "parametrize" and m.args[0] == names)


KERNELS = [("sdpa_flash", {"sdpa_narrow": 0}), ("sdpa_narrow", {"sdpa_narrow": 2}), ("sdpa_narrow", {"sdpa_narrow": 2, "sdpa_narrow_split": 1}),
           ("sdpa_narrow", {"sdpa_narrow": 2, "sdpa_narrow_split": 2}), ("sdpa_narrow", {"sdpa_narrow": 2, "sdpa_narrow_split": 4})]
kernels = pytest.mark.parametrize("kernel,options", KERNELS, ids=["flash", "narrow", "narrow1", "narrow2", "narrow4"])


@kernels
@pytest.mark.parametrize("dtype", [W.F16, W.BF16])
@pytest.mark.parametrize("shape,causal", parameters(parity.test_sdpa_flash, "shape,causal"))
def test_shapes(hip, oracle, schedule_options, kernel, options, dtype, shape, causal):
    schedule_options(options)
    parity.test_sdpa_flash(hip, oracle, dtype, shape, causal)
    assert hip.last_sdpa_kernel() == kernel


@kernels
@pytest.mark.parametrize("dtype", [W.F16, W.BF16])
@pytest.mark.parametrize("profile", ["ramp", "step16", "step40", "spike", "fall", "wide"])
def test_scores_that_grow_along_the_keys(hip, oracle, schedule_options, kernel, options, dtype, profile):
    schedule_options(options)
    for causal in (False, True):
        parity.test_sdpa_flash_scores_that_grow_along_the_keys(hip, oracle, dtype, profile, causal)
        assert hip.last_sdpa_kernel() == kernel


@kernels
@pytest.mark.parametrize("D", [128, 96, 72])
@pytest.mark.parametrize("dtype", [W.F16, W.BF16])
@pytest.mark.parametrize("kind", parity.FLASH_MASKS)
def test_masks(hip, oracle, schedule_options, kernel, options, dtype, kind, D):
    schedule_options(options)
    for shape in parameters(parity.test_sdpa_flash_with_mask, "B,Hq,Hkv,Lq,Lk"):
        parity.test_sdpa_flash_with_mask(hip, oracle, dtype, kind, *shape, D)
        rides = shape[4] % (16 if kind.startswith("bool") else 8) == 0  # (the head-128 kernel wants aligned mask rows)
        assert hip.last_sdpa_kernel() == (kernel if rides or kernel == "sdpa_narrow" else "sdpa_flash_small")


@pytest.mark.parametrize("narrow_option", [0, 2])
@pytest.mark.parametrize("seed", [21, 22])
def test_random_shapes(hip, oracle, schedule_options, seed, narrow_option):
    schedule_options({"sdpa_narrow": narrow_option})
    random_tests.test_random_sdpa_shapes(hip, oracle, seed)


@pytest.mark.parametrize("split", [1, 2, 4])
@pytest.mark.parametrize("dtype", [W.F16, W.BF16])
@pytest.mark.parametrize("mask", ["none", "causal", "padding", "scattered", "bias"])
def test_narrow_shapes_by_split(hip, oracle, schedule_options, mask, dtype, split):
    """The shapes of the narrow kernel's own tests, and key counts of ten tiles and more, past which every stage of its pipeline has
    been used again."""
    schedule_options({"sdpa_narrow": 2, "sdpa_narrow_split": split})
    for shape in narrow.SHAPES + [(1, 2, 1, 70, 700, 64), (1, 2, 2, 40, 641, 96), (1, 2, 1, 33, 1000, 128), (2, 2, 2, 130, 672, 80), (1, 1, 1, 300, 1301, 64)]:
        narrow.test_sdpa_narrow(hip, oracle, shape, mask, dtype)
        assert hip.last_sdpa_kernel() == "sdpa_narrow" or shape[4] == 1  # (a mask of one key is broadcast: stride 0)


@pytest.mark.parametrize("split", [1, 2, 4])
@pytest.mark.parametrize("dtype", [W.F16, W.BF16])
def test_narrow_references_by_split(hip, oracle, schedule_options, dtype, split):
    """References that move: along growing scores, on masks of the lowest value, with constants added to the rows."""
    schedule_options({"sdpa_narrow": 2, "sdpa_narrow_split": split})
    narrow.test_growing_scores(hip, oracle, dtype)
    for shape in parameters(narrow.test_masks_of_the_lowest_value, "shape"):
        narrow.test_masks_of_the_lowest_value(hip, oracle, dtype, shape)
    for shape in [(1, 4, 2, 130, 400, 64), (1, 4, 2, 130, 400, 96), (1, 4, 2, 130, 400, 128), (1, 4, 4, 130, 203, 72), (1, 2, 2, 130, 401, 120)]:
        narrow.test_a_constant_added_to_a_row_changes_nothing(hip, oracle, dtype, shape)


@pytest.mark.parametrize("profile", ["ramp", "step", "late"])
@pytest.mark.parametrize("split", [1, 2, 4])
@pytest.mark.parametrize("dtype", [W.F16, W.BF16])
@pytest.mark.parametrize("D", [64, 96, 128])
def test_late_moves_of_the_reference(hip, oracle, schedule_options, D, dtype, split, profile):
    """Scores that leave what the sums allow after many tiles, in the first and in the second half of one: what was summed up and
    the scores already under way move along.  Column 0 carries the growth, in powers of two that the type represents, so
    that the oracle's scores have it too and differ by the other columns' rounding alone."""
    schedule_options({"sdpa_narrow": 2, "sdpa_narrow_split": split})
    case = W.make_sdpa_case(25, 1, 2, 2, 70, 600, D, dtype, std=0.5 if dtype == W.BF16 else 1.0)
    keys = np.arange(600)
    growth = {"ramp": keys // 8 * 2.0, "step": np.where(keys >= 399, 64.0, 0.0), "late": np.where(keys % 200 == 170, 32.0 + keys // 200 * 32.0, 0.0)}[profile]
    scale = 0.125  # (so that q * scale is a power of two in column 0)
    case["q"][..., 0], case["k"][..., 0] = 2.0, growth
    for n in "qk":
        case[n + "_store"], case[n] = W.to_storage(case[n], dtype)
    out, _ = H.run_sdpa(hip, case, False, scale=scale)
    assert hip.last_sdpa_kernel() == "sdpa_narrow"
    ref = oracle.sdpa(case["q"], case["k"], case["v"], scale=scale)
    # q * scale * log2(e) is rounded to 16 bits: scores of up to 150 / 8 * 2 = 37 nats lose up to 37 * 2^-12 (2^-9) together, and
    # their differences among keys that count, within 8 nats of the top, 8 * 2^-12 (2^-9), on values up to 4
    assert np.isfinite(out).all()
    assert H.scaled_bound_error(out, ref, "late moves") <= (8e-3 if dtype == W.F16 else 6.4e-2)


@pytest.mark.parametrize("shape", [(1, 72, 9, 300, 300, 64), (3, 24, 8, 200, 200, 96), (1, 104, 13, 140, 140, 128), (1, 136, 17, 97, 97, 64)])
@pytest.mark.parametrize("split", [1, 2, 4])
def test_causal_heads_in_groups(hip, oracle, schedule_options, shape, split):
    """Causal calls hand out the longest tiles of eight heads first: more than eight heads to an XCD, the last group not full."""
    schedule_options({"sdpa_narrow": 2, "sdpa_narrow_split": split})
    B, Hq, Hkv, Lq, Lk, D = shape
    case = W.make_sdpa_case(26, B, Hq, Hkv, Lq, Lk, D, W.F16)
    out, _ = H.run_sdpa(hip, case, True)
    assert np.isfinite(out).all()
    assert H.scaled_bound_error(out, oracle.sdpa(case["q"], case["k"], case["v"], causal=True), "causal groups") <= TOL[W.F16]


# what the rule picks for large calls: one wavefront to 32 rows, more than one round of workgroups
@pytest.mark.parametrize("mask", ["none", "causal", "padding", "bias"])
@pytest.mark.parametrize("shape", [(8, 32, 8, 257, 577, 64), (4, 32, 8, 257, 400, 96), (4, 32, 32, 130, 330, 128)])
def test_large_unsplit_calls(hip, oracle, schedule_options, shape, mask):
    schedule_options({"sdpa_narrow": 2})
    narrow.test_sdpa_narrow(hip, oracle, shape, mask, W.F16)
    assert hip.last_sdpa_kernel() == "sdpa_narrow"


class Shifted:
    """A device copy of an array that starts `offset` bytes behind a 256-byte boundary."""

    def __init__(self, hip, array, offset):
        import ctypes

        self.array, self.offset, self.nbytes = array, offset, array.nbytes
        raw = np.zeros(array.nbytes + 256, np.uint8)
        raw[offset:offset + array.nbytes] = np.ascontiguousarray(array).view(np.uint8).ravel()
        self.buffer = hip.DeviceBuffer.from_numpy(raw)
        self.ptr = ctypes.c_void_p(self.buffer.ptr.value + offset)

    def download(self):
        raw = self.buffer.download(np.uint8, (self.nbytes + 256,))[self.offset:self.offset + self.nbytes]
        return np.frombuffer(raw.tobytes(), self.array.dtype).reshape(self.array.shape)


@pytest.mark.parametrize("mask", ["none", "causal", "bool", "bias"])
@pytest.mark.parametrize("dtype", [W.F16, W.BF16])
def test_operands_off_16_bytes(hip, oracle, dtype, mask):
    """Head size 128 with operands that start eight bytes behind a multiple of 16: the tuned head-128 kernel takes them."""
    B, Hq, Hkv, Lq, Lk, D = 1, 4, 2, 150, 208, 128
    case = W.make_sdpa_case(27, B, Hq, Hkv, Lq, Lk, D, dtype)
    bufs = [Shifted(hip, case[n + "_store"], 8) for n in "qkv"]
    out = Shifted(hip, np.full_like(case["q_store"], 0xFFFF), 8)
    desc = hip.SdpaDesc(dtype, B, Hq, Hkv, Lq, Lk, D, int(mask == "causal"), 0.0)
    rng = np.random.default_rng(5)
    if mask in ("none", "causal"):
        hip.sdpa(desc, *bufs, out)
        ref = oracle.sdpa(case["q"], case["k"], case["v"], causal=mask == "causal")
    else:
        m = rng.random((Lq, Lk)) < 0.6 if mask == "bool" else W.to_storage(rng.standard_normal((Lq, Lk)).astype(np.float32), dtype)[1]
        m[..., 0] = 1
        store = m.astype(np.uint8) if mask == "bool" else W.to_storage(m, dtype)[0]
        hip.sdpa_masked(desc, *bufs, W.U8 if mask == "bool" else dtype, [0, 0, Lk, 1], hip.DeviceBuffer.from_numpy(store), out)
        ref = oracle.sdpa_masked(case["q"], case["k"], case["v"], m)
    assert hip.last_sdpa_kernel() == "sdpa_flash"
    got = H.storage_to_f32(out.download(), dtype)
    assert np.isfinite(got).all()
    assert H.scaled_bound_error(got, ref, "off 16 bytes") <= TOL[dtype]


def test_which_kernel_the_rule_takes(hip, oracle):
    """Calls on either side of the lines the rules draw."""
    for (B, Hq, Hkv, Lq, Lk, D, dtype, causal), kernel in [
            ((1, 4, 4, 64, 64, 64, W.F16, False), "sdpa_narrow"), ((1, 4, 4, 64, 64, 96, W.BF16, True), "sdpa_narrow"),
            ((1, 8, 8, 48, 48, 128, W.F16, True), "sdpa_narrow"), ((4, 32, 8, 1024, 1024, 128, W.BF16, True), "sdpa_flash"),
            ((2, 12, 12, 1390, 1390, 80, W.F16, False), "sdpa_flash"), ((2, 12, 12, 1390, 1390, 80, W.F16, True), "sdpa_narrow"),
            ((1, 4, 4, 64, 64, 56, W.F16, False), "sdpa_flash"), ((1, 4, 4, 64, 64, 256, W.F16, False), "sdpa_flash_small"),
            ((1, 4, 4, 64, 64, 64, W.F32, False), "sdpa_f32"), ((1, 4, 4, 64, 64, 136, W.F32, False), "sdpa_generic")]:
        H.run_sdpa(hip, W.make_sdpa_case(28, B, Hq, Hkv, Lq, Lk, D, dtype), causal)
        assert hip.last_sdpa_kernel() == kernel, (B, Hq, Lq, D, dtype)
