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
