"""Infinities and NaN where kernels treat them apart: the direct matrix-core
kernel computes such workgroups anew in the reference's order (a sample under
a zero tap does not count)."""
import numpy as np
import pytest

import ndconv as nc
from modes import conv_mode, padding_mode
from oracle import ndconv_oracle as O

pytestmark = pytest.mark.gpu


# small kernels, whose recomputation takes a wave less time than another wave's
# products, over tiles of 16, 32 and 64 rows; bars as in test_matrix_gpu.py
@pytest.mark.parametrize("algo", ["auto", "bf16", "bf16x3"])
@pytest.mark.parametrize("ks", [(1, 1), (1, 2), (3, 3), (1, 33)])
@pytest.mark.parametrize("shape", [(40, 270), (700, 600), (2600, 2100)])
def test_direct_matrix_small_kernels(gpu, shape, ks, algo):
    rng = np.random.default_rng(ks[0] * 100 + ks[1])
    x = rng.standard_normal(shape).astype(np.float32)
    k = rng.standard_normal(ks).astype(np.float32)
    if k.size > 1:
        k.flat[k.size // 2] = 0.0
    h, w = shape
    for i, j, v in [(0, 0, np.nan), (1, 200, np.inf), (h // 2, 255, -np.inf), (h // 2, 256, np.inf), (h - 1, w - 1, np.nan),
                    (h // 3, w // 3, np.inf), (h - 2, 3, -np.inf)]:
        x[i, j] = v
    with np.errstate(invalid="ignore"):
        ref = O.conv(x, k, "same", "replicate")                           # float32, offset-list order
        ref64 = O.conv(x, k, "same", "replicate", acc_dtype=np.float64)
    fin = np.isfinite(ref64)
    assert 0 < fin.sum() < fin.size
    for _ in range(3):
        got = nc.conv(x, k, conv_mode("same"), padding_mode("replicate"), algo=algo)
        np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
        np.testing.assert_array_equal(np.isposinf(got), np.isposinf(ref))
        np.testing.assert_array_equal(np.isneginf(got), np.isneginf(ref))
        assert O.relerr(got[fin], ref64[fin])[0] <= (1e-2 if algo == "bf16" else 1e-5)
