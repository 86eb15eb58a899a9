"""Products of 7 to 64 rows with weights stored [n, k], against the oracle: both sides of every tile of 16 rows, weight rows that do
not fill a workgroup's, one stage of k to several rounds of the ring, k whole and in parts (with the workspace that parts need), and a
k that is no whole stage (the library's).  Bound: that of the general matmul test, one rounding of the result and 1e-6 sqrt(k) for the
fp32 sum of k products."""
import numpy as np
import pytest

from test_gpu_layer_ops import BF16, F16, F32, ROUND, download, ops, scaled_error, upload  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("m,n,k", [(7, 4, 64), (16, 100, 4160), (17, 1024, 4096), (32, 6144, 320), (33, 68, 704), (48, 512, 640), (49, 4096, 1024), (64, 128, 14336),
                                   (64, 22016, 128), (20, 6160, 768), (64, 36, 8192), (12, 5500, 192), (40, 64, 96), (50, 33000, 64), (30, 28676, 320)])
def test_matmul_mid_rows(hip, ops, oracle, m, n, k, dtype):  # noqa: F811
    rng = np.random.default_rng(m + n + k)
    da, a = upload(hip, rng.standard_normal((1, m, k)) * 0.5, dtype)
    db, b = upload(hip, rng.standard_normal((n, k)) * 0.5, dtype)
    ref = oracle.matmul(a, b, False, True)
    d = ops.MatmulDesc(dtype, dtype, m, n, k, 1, 0, 1, 0, 0)
    workspace = hip.DeviceBuffer(ops.matmul_workspace_size(d))
    workspace.fill(0xFF)
    for c_dtype, ws in ((dtype, workspace), (F32, workspace), (dtype, None)):
        dc = hip.DeviceBuffer(m * n * hip.DTYPE_BYTES[c_dtype])
        dc.fill(0xFF)
        ops.matmul(ops.MatmulDesc(dtype, c_dtype, m, n, k, 1, 0, 1, 0, 0), da, db, dc, ws)
        got = download(hip, dc, c_dtype, (1, m, n))
        assert scaled_error(got, ref) <= (ROUND[dtype] if c_dtype == dtype else 0) + 1e-6 * np.sqrt(k)


@pytest.mark.parametrize("m,n,k", [(16, 2816, 5120), (17, 2816, 5120), (16, 2812, 5120), (8, 4096, 9216), (8, 4096, 9280), (16, 6144, 3072), (32, 7168, 5120), (33, 8192, 4096),
                                   (32, 512, 2048), (32, 512, 2112), (33, 512, 1536), (33, 512, 1600), (64, 11008, 2048), (64, 11004, 2048)])
def test_matmul_either_side_of_the_library(hip, ops, oracle, m, n, k):  # noqa: F811
    """Sizes either side of the lines between the library and the kernel of few rows, with the workspace, with room for two parts of k and without."""
    rng = np.random.default_rng(m + n + k)
    da, a = upload(hip, rng.standard_normal((1, m, k)) * 0.5, BF16)
    db, b = upload(hip, rng.standard_normal((n, k)) * 0.5, BF16)
    ref = oracle.matmul(a, b, False, True)
    d = ops.MatmulDesc(BF16, BF16, m, n, k, 1, 0, 1, 0, 0)
    for ws in (hip.DeviceBuffer(ops.matmul_workspace_size(d)), hip.DeviceBuffer(2 * m * n * 4), None):
        dc = hip.DeviceBuffer(m * n * 2)
        dc.fill(0xFF)
        ops.matmul(d, da, db, dc, ws)
        assert scaled_error(download(hip, dc, BF16, (1, m, n)), ref) <= ROUND[BF16] + 1e-6 * np.sqrt(k)


def test_long_k_without_a_workspace_is_not_one_chain(hip, ops):  # noqa: F811
    """Without room for parts of k a workgroup would walk all of it (64 rows, 16 x 16,384: 75 us against 10 with the workspace and 14 in the library)."""
    m, n, k = 64, 16, 16384
    d = ops.MatmulDesc(BF16, BF16, m, n, k, 1, 0, 1, 0, 0)
    a, b, c = hip.DeviceBuffer(m * k * 2), hip.DeviceBuffer(n * k * 2), hip.DeviceBuffer(m * n * 2)
    a.fill(0)
    b.fill(0)
    before, after = hip.Event(), hip.Event()
    times = []
    for ws in (hip.DeviceBuffer(ops.matmul_workspace_size(d)), None):
        best = float("inf")
        for _ in range(5):  # (the first of them chooses the library's algorithm)
            before.record()
            for _ in range(50):
                ops.matmul(d, a, b, c, ws)
            after.record()
            after.synchronize()
            best = min(best, before.elapsed_ms(after))
        times.append(best)
    assert times[1] <= 3 * times[0], times
