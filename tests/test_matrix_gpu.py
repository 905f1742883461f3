"""Direct rank-2 convolutions on the matrix cores (matrix_conv.hip) and the
staged direct kernel against the oracle: outputs one short of, equal to and
one past whole tiles (16, 32 and 64 rows of 256 columns), kernel widths on
both sides of every operand block, phases of a dilated axis, decimated input,
every border, full-range integers (exact) and views.  Tolerances are the
suite's bars: 1e-5 for f32 and BF16x3, 1e-2 for BF16, 1e-12 for f64."""
import numpy as np
import pytest

import ndconv as nc
from modes import conv_mode, padding_mode
from oracle import ndconv_oracle as O

pytestmark = pytest.mark.gpu


def rand(rng, shape, dtype):
    dt = np.dtype(dtype)
    if dt.kind == "c":
        return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(dt)
    if dt.kind == "f":
        return rng.standard_normal(shape).astype(dt)
    i = np.iinfo(dt)   # the whole range: every byte of every value counts
    return rng.integers(i.min, i.max, shape, dtype=dt, endpoint=True)


def check(x, k, mode="same", pm="zeros", dil=1, rev=True, algo="auto"):
    kw = nc.with_dilation(k, dil)
    got = nc.conv(x, kw if rev else kw.no_reverse(), conv_mode(mode), padding_mode(pm), algo=algo)
    if x.dtype.kind in "iu":
        np.testing.assert_array_equal(got, O.conv(x, k, mode, pm, dil, rev))
        return
    wide = np.complex128 if x.dtype.kind == "c" else np.float64
    ref = O.conv(x.astype(wide), k.astype(wide), mode, pm, dil, rev)
    tol = 1e-2 if algo == "bf16" else 1e-12 if x.dtype.itemsize // (2 if x.dtype.kind == "c" else 1) == 8 else 1e-5
    assert got.shape == ref.shape
    assert O.relerr(got, ref)[0] <= tol


INTS = [np.int8, np.uint8, np.int16, np.uint16, np.int32, np.uint32, np.int64, np.uint64]


@pytest.mark.parametrize("dtype", INTS + [np.float32, np.float64, np.complex64])
@pytest.mark.parametrize("shape", [(1, 1), (15, 255), (16, 256), (17, 257), (33, 300), (65, 513), (3, 1000)])
def test_tile_edges(gpu, dtype, shape):
    rng = np.random.default_rng(shape[0] + shape[1])
    k = rand(rng, (min(3, shape[0]), min(5, shape[1])), dtype)
    check(rand(rng, shape, dtype), k, "same", "zeros")
    check(rand(rng, shape, dtype), k, "full", "replicate", 1, False)


@pytest.mark.parametrize("kw", [1, 2, 3, 4, 7, 8, 15, 17, 18, 27, 31, 32, 39, 40, 47, 48, 49, 50])
@pytest.mark.parametrize("dtype,algo", [(np.float32, "auto"), (np.float32, "bf16x3"), (np.float32, "bf16"),
                                        (np.int32, "auto"), (np.int16, "auto"), (np.float64, "auto")])
def test_kernel_widths(gpu, dtype, algo, kw):
    rng = np.random.default_rng(kw)
    kh = 5 if kw < 30 else 9
    check(rand(rng, (40, 270), dtype), rand(rng, (kh, kw), dtype), "valid", "zeros", 1, True, algo)


@pytest.mark.parametrize("kh", [1, 2, 4, 5, 31, 33, 64, 100])
@pytest.mark.parametrize("dtype,algo", [(np.float32, "auto"), (np.float32, "bf16x3"), (np.int32, "auto")])
def test_kernel_heights(gpu, dtype, algo, kh):
    rng = np.random.default_rng(kh)
    k = rand(rng, (kh, 33 if algo == "bf16x3" else 7), dtype)
    check(rand(rng, (130, 70), dtype), k, "valid", "zeros", 1, True, algo)


BORDERS = ["zeros", ("const", 3), "reflect", "replicate", "circular", ("custom", [("const", 2), "circular"]),
           ("explicit", [[("const", 1), ("const", 5)], ["circular", "reflect"]])]


@pytest.mark.parametrize("dtype,algo", [(np.float32, "auto"), (np.float32, "bf16x3"), (np.int32, "auto"),
                                        (np.uint8, "auto"), (np.float64, "auto")])
@pytest.mark.parametrize("pm", BORDERS)
@pytest.mark.parametrize("strides,dil", [([1, 1], [1, 1]), ([1, 1], [3, 2]), ([2, 2], [2, 2]), ([1, 3], [2, 3]),
                                         ([2, 1], [4, 2]), ([2, 3], [2, 1])])
def test_borders_strides_dilations(gpu, dtype, algo, pm, strides, dil):
    rng = np.random.default_rng(9)
    args = (rand(rng, (60, 290), dtype), rand(rng, (6, 7), dtype), ("explicit", [[5, 9], [11, 4]], strides), pm, dil, False,
            algo)
    if algo == "bf16x3" and strides == [2, 3]:   # rows of 128 outputs at stride 3 and dilation 1 exceed the staged width
        with pytest.raises(nc.Unsupported):
            check(*args)
        return
    check(*args)


@pytest.mark.parametrize("dil,refused", [([1, 8], False), ([1, 9], True), ([5, 1], True), ([4, 1], False)])
def test_bf16_refusals(gpu, dil, refused):
    rng = np.random.default_rng(10)
    x, k = rand(rng, (90, 300), np.float32), rand(rng, (6, 7), np.float32)
    if refused:
        with pytest.raises(nc.Unsupported):
            check(x, k, "same", "zeros", dil, True, "bf16x3")
    else:
        check(x, k, "same", "zeros", dil, True, "bf16x3")


def test_views(gpu):
    rng = np.random.default_rng(12)
    for dt in (np.float32, np.int32, np.int16, np.float64):
        x, k = rand(rng, (310, 260), dt), rand(rng, (14, 18), dt)
        for xv, kv in [(x.T, k), (x[::-1], k[:, ::-1]), (x[::2, ::-3], k[::-2, ::2]), (x[5:200, 7:30], k.T[:3, :2])]:
            check(xv, kv, "same", "reflect")
    x = rand(rng, (6, 20, 30), np.float64)
    check(x[::-1, :, ::-1], rand(rng, (2, 3, 4), np.float64), "full", ("custom", [("const", 2.0), "reflect", "circular"]))
    check(rand(rng, (500,), np.float32)[::-2], rand(rng, (9,), np.float32), "same", "circular")


def test_bf16x3_of_few_taps_is_exact(gpu):
    """Fewer than 32 taps: the FP32 kernel, bit for bit."""
    rng = np.random.default_rng(14)
    x, k = rand(rng, (70, 300), np.float32), rand(rng, (4, 7), np.float32)
    y = [nc.conv(x, k, nc.ConvMode.Same, nc.PaddingMode.Zeros, algo=a) for a in ("auto", "bf16x3")]
    np.testing.assert_array_equal(y[0], y[1])
