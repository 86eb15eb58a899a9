"""Products of up to 16 rows with weights stored [n, k], against the oracle: one row to all sixteen and one more, weight
rows that do not fill a tile of 16, fewer steps of k than wavefronts, and a last round of loads that is not full.
Bound: that of the general matmul test, one rounding of the result and 1e-6 sqrt(k) for the fp32 sum of k products."""
import numpy as np
import pytest

from test_gpu_layer_ops import BF16, F16, F32, ROUND, download, ops, scaled_error, upload  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("m,n,k", [(1, 4, 32), (1, 1024, 4096), (3, 20, 96), (4, 4096, 2080), (7, 36, 256), (16, 128, 14336), (15, 52, 8192), (6, 8196, 2048), (6, 8200, 2080),
                                   (17, 64, 512), (5, 30, 128), (2, 64, 72)])
def test_matmul_few_rows(hip, ops, oracle, m, n, k, dtype):  # noqa: F811
    rng = np.random.default_rng(m + n + k)
    da, a = upload(hip, rng.standard_normal((1, m, k)) * 0.5, dtype)
    db, b = upload(hip, rng.standard_normal((n, k)) * 0.5, dtype)
    ref = oracle.matmul(a, b, False, True)
    for c_dtype in (dtype, F32):
        dc = hip.DeviceBuffer(m * n * hip.DTYPE_BYTES[c_dtype])
        dc.fill(0xFF)
        ops.matmul(ops.MatmulDesc(dtype, c_dtype, m, n, k, 1, 0, 1, 0, 0), da, db, dc, None)
        got = download(hip, dc, c_dtype, (1, m, n))
        assert scaled_error(got, ref) <= (ROUND[dtype] if c_dtype == dtype else 0) + 1e-6 * np.sqrt(k)


# either side of where the rule leaves a long k to the library: any n, n against k, and 16 rows
@pytest.mark.parametrize("m,n,k", [(6, 16, 6144), (6, 16, 6176), (4, 2048, 7168), (4, 2044, 7168), (16, 64, 4096), (16, 64, 4128)])
def test_matmul_lines_of_the_rule(hip, ops, oracle, m, n, k):  # noqa: F811
    test_matmul_few_rows(hip, ops, oracle, m, n, k, BF16)
