"""Infinities and NaN where kernels treat them apart: the direct matrix-core
kernel computes such workgroups in the reference's order (a sample under a
zero tap does not count); conv_fft gives NaN everywhere, also for a value that
no tile reads."""
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


def spread(x, k, mode, pm, dil, baked):
    """All NaN for x and k as the oracle has it, and finite for the call after."""
    kv = nc.with_dilation(k, dil)
    m, p = conv_mode(mode), padding_mode(pm)
    with np.errstate(invalid="ignore"):
        assert not np.isfinite(O.conv_fft(x.astype(np.float64), k.astype(np.float64), mode, pm, dil)).any()
    got = nc.conv_fft_with_baked(x, nc.conv_fft_bake(x, kv, m, p)) if baked else nc.conv_fft(x, kv, m, p)
    assert np.isnan(got).all()
    y = nc.conv_fft(np.ones(x.shape, x.dtype), nc.with_dilation(np.ones(k.shape, k.dtype), dil), m, nc.PaddingMode.Zeros)
    assert np.isfinite(y).all()


# planes between the taps of a stride or dilation, and past the last output; x
# of kept spectra (small) and transformed per tap (large, or a constant border)
@pytest.mark.parametrize("baked", [False, True])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("pm", ["zeros", "circular", ("const", 0.5)])
@pytest.mark.parametrize("shape,ks,strides,dil,plane", [
    ((9, 40, 50), (2, 3, 5), [2, 1, 1], [2, 1, 1], 1), ((9, 40, 50), (1, 3, 5), [3, 1, 1], 1, 8),
    ((10, 30, 41), (3, 3, 3), [2, 2, 1], 1, 9), ((7, 40, 50), (2, 3, 5), [1, 1, 1], [5, 1, 1], 3),
    ((40, 200, 260), (3, 3, 3), [4, 1, 1], 1, 3)])
def test_planes_between_taps(gpu, shape, ks, strides, dil, plane, pm, dtype, baked):
    rng = np.random.default_rng(6)
    x, k = rng.standard_normal(shape).astype(dtype), rng.standard_normal(ks).astype(dtype)
    for v, i, j in ((np.nan, 0, 0), (np.inf, shape[1] - 1, shape[2] - 1)):
        bad = x.copy()
        bad[plane, i, j] = v
        spread(bad, k, ("explicit", [[0, 0], [1, 1], [1, 1]], strides), pm, dil, baked)


@pytest.mark.parametrize("baked", [False, True])
@pytest.mark.parametrize("shape,ks", [((1, 40, 50), (3, 3, 5)), ((2, 3, 30, 40), (5, 1, 3, 3)), ((1, 900, 1200), (3, 3, 3))])
def test_taps_that_meet_zeros_only(gpu, shape, ks, baked):
    rng = np.random.default_rng(7)
    x, k = rng.standard_normal(shape).astype(np.float32), rng.standard_normal(ks).astype(np.float32)
    for i in (0, k.size - 1):
        bad = k.copy()
        bad.flat[i] = np.inf
        spread(x, bad, "same", "zeros", 1, baked)


# one launch, tiles, kept spectra; a plane of fill that a stride steps over
@pytest.mark.parametrize("baked", [False, True])
@pytest.mark.parametrize("v", [np.inf, np.nan, 1e300])
@pytest.mark.parametrize("shape,ks,mode", [((5000,), (31,), "same"), ((50000,), (31,), "full"), ((90, 300), (5, 7), "same"),
                                           ((6, 50, 60), (1, 3, 3), ("explicit", [[1, 1], [1, 1], [1, 1]], [3, 1, 1]))])
def test_nonfinite_constant(gpu, shape, ks, mode, v, baked):
    rng = np.random.default_rng(8)
    x, k = rng.standard_normal(shape).astype(np.float32), rng.standard_normal(ks).astype(np.float32)
    v32 = float(np.float32(v)) if v != 1e300 else np.inf   # what the constant is in f32
    pm = ("const", v)
    kv, m = nc.with_dilation(k, 1), conv_mode(mode)
    with np.errstate(invalid="ignore"):
        assert not np.isfinite(O.conv_fft(x.astype(np.float64), k.astype(np.float64), mode, ("const", v32))).any()
    p = padding_mode(pm)
    got = nc.conv_fft_with_baked(x, nc.conv_fft_bake(x, kv, m, p)) if baked else nc.conv_fft(x, kv, m, p)
    assert np.isnan(got).all()
    assert np.isfinite(nc.conv_fft(x, kv, m, nc.PaddingMode.Zeros)).all()
