"""conv_fft by overlap-save tiles against the FP64 oracle, at the sizes where a
tile can go wrong: outputs one short of, equal to and one past a whole number
of tiles, single and odd tile counts, phases of unequal length, and every form
of view, border and option the tiles accept.  Tolerances are the suite's bars
(1e-5 single, 1e-12 double precision); a tile's transform is shorter than the
whole-array one these were set for."""
import numpy as np
import pytest

import ndconv as nc
from modes import conv_mode, padding_mode, rand_array
from oracle import ndconv_oracle as O

pytestmark = pytest.mark.gpu

TOL = {np.dtype(np.float32): 1e-5, np.dtype(np.complex64): 1e-5, np.dtype(np.float64): 1e-12,
       np.dtype(np.complex128): 1e-12}


def wide(a):
    return a.astype(np.complex128 if a.dtype.kind == "c" else np.float64)


def check(x, k, mode="same", pm="zeros", dil=1, rev=True):
    kw = nc.with_dilation(k, dil)
    got = nc.conv_fft(x, kw if rev else kw.no_reverse(), conv_mode(mode), padding_mode(pm))
    ref = O.conv_fft(wide(x), wide(k), mode, pm, dil, rev)
    assert got.shape == ref.shape
    assert O.relerr(got, ref)[0] <= TOL[x.dtype]
    return got


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64, np.complex128])
@pytest.mark.parametrize("n,k", [(1, 1), (993, 31), (994, 31), (995, 31), (1987, 31), (1988, 31), (1989, 31), (4000, 31),
                                 (16384, 31), (16385, 31), (20000, 1024), (9000, 1500), (40000, 2500)])
def test_rank1_edges(gpu, dtype, n, k):
    rng = np.random.default_rng(n + k)
    k = min(k, n)
    check(rand_array(rng, n, dtype), rand_array(rng, k, dtype), "same", "reflect" if n > k else "zeros")


@pytest.mark.parametrize("k", [6000, 12000])
def test_rank1_long_kernel(gpu, k):
    rng = np.random.default_rng(k)
    check(rand_array(rng, 60001, np.float32), rand_array(rng, k, np.float32), "valid", "zeros", 1, False)


# the outputs of 32x32, 32x128, 64x64, 64x128 and 128x128 tiles, whole and one off
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64])
@pytest.mark.parametrize("shape,k", [((30, 30), (3, 3)), ((31, 61), (3, 3)), ((44, 196), (11, 31)), ((45, 197), (11, 31)),
                                     ((300, 400), (21, 25)), ((301, 399), (31, 31)), ((513, 700), (31, 31)),
                                     ((1200, 900), (9, 41)), ((1100, 1100), (70, 50)), ((1, 3000), (1, 63)),
                                     ((3000, 1), (63, 1)), ((7, 5), (7, 5))])
def test_rank2_edges(gpu, dtype, shape, k):
    rng = np.random.default_rng(shape[0] * 7 + shape[1])
    check(rand_array(rng, shape, dtype), rand_array(rng, k, dtype), "full", "zeros")
    check(rand_array(rng, shape, dtype), rand_array(rng, k, dtype), "same", "replicate", 1, False)


BORDERS = ["zeros", ("const", 0.75), "reflect", "replicate", "circular",
           ("custom", [("const", -1.5), "circular"]), ("custom", ["reflect", ("const", 2.0)]),
           ("explicit", [[("const", 1.0), ("const", -2.0)], ["circular", "reflect"]])]


@pytest.mark.parametrize("dtype", [np.float32, np.complex128])
@pytest.mark.parametrize("pm", BORDERS)
@pytest.mark.parametrize("mode,dil", [("full", 1), ("same", [2, 3]), (("custom", [5, 9], [2, 3]), [1, 2]),
                                      (("explicit", [[3, 0], [1, 12]], [1, 2]), 2)])
def test_borders_and_options(gpu, dtype, pm, mode, dil):
    rng = np.random.default_rng(3)
    check(rand_array(rng, (75, 130), dtype), rand_array(rng, (5, 8), dtype), mode, pm, dil, rev=mode == "full")


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64])
@pytest.mark.parametrize("pm", ["zeros", "circular", ("custom", [("const", 3.0), "reflect", ("const", -1.0)])])
@pytest.mark.parametrize("shape,k", [((5, 40, 90), (3, 5, 9)), ((9, 70, 33), (2, 9, 4)), ((2, 3, 40, 41), (2, 2, 3, 3))])
def test_outer_taps(gpu, dtype, pm, shape, k):
    if len(shape) == 4 and not isinstance(pm, str):
        pm = ("custom", [("const", 3.0), "replicate", ("const", -1.0), "circular"])
    rng = np.random.default_rng(len(shape))
    x, kv = rand_array(rng, shape, dtype), rand_array(rng, k, dtype)
    check(x, kv, "full", pm)
    check(x, kv, ("custom", [1] * len(shape), [2] + [1] * (len(shape) - 1)), pm, [2] + [1] * (len(shape) - 1), False)


def test_views(gpu):
    """Transposed, reversed and stepped views of x and k."""
    rng = np.random.default_rng(11)
    x, k = rand_array(rng, (310, 260), np.float32), rand_array(rng, (14, 18), np.float32)
    for xv, kv in [(x.T, k), (x[::-1], k[:, ::-1]), (x[::2, ::-3], k[::-2, ::2]), (x[5:200, 7:9], k.T[:3, :2]),
                   (np.broadcast_to(x[:1], (90, 260)), k)]:
        check(xv, kv, "same", "reflect" if min(xv.shape) > 20 else "zeros")
    check(x[::-1, 3], k[::-1, 2], "full", "circular")


@pytest.mark.parametrize("shape,k", [((3000,), (31,)), ((50000,), (31,)), ((90, 300), (5, 7)), ((6, 50, 60), (2, 3, 3))])
def test_nonfinite_spreads_and_clears(gpu, shape, k):
    """One non-finite value makes the whole result NaN, and the next call clean."""
    rng = np.random.default_rng(5)
    x, kv = rand_array(rng, shape, np.float32), rand_array(rng, k, np.float32)
    for v in (np.inf, -np.inf, np.nan):
        for i in (0, x.size // 2, x.size - 1):
            bad = x.copy()
            bad.flat[i] = v
            assert np.isnan(nc.conv_fft(bad, kv, nc.ConvMode.Same, nc.PaddingMode.Zeros)).all()
    bad = kv.copy()
    bad.flat[0] = np.inf
    assert np.isnan(nc.conv_fft(x, bad, nc.ConvMode.Same, nc.PaddingMode.Zeros)).all()
    check(x, kv)


@pytest.mark.parametrize("shape,k", [((3000,), (31,)), ((50000,), (1031,)), ((90, 300), (5, 7)), ((6, 50, 60), (2, 3, 3))])
def test_baked_is_the_same(gpu, shape, k):
    rng = np.random.default_rng(6)
    x, kv = rand_array(rng, shape, np.float32), rand_array(rng, k, np.float32)
    b = nc.conv_fft_bake(x, kv, nc.ConvMode.Same, nc.PaddingMode.Circular)
    y = nc.conv_fft(x, kv, nc.ConvMode.Same, nc.PaddingMode.Circular)
    np.testing.assert_array_equal(nc.conv_fft_with_baked(x, b), y)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_processor_after_other_kernels(gpu, dtype):
    """The inverse transform's first reads of the factors it stages in LDS,
    where another kernel has left other values."""
    rng = np.random.default_rng(8)
    x, k = rand_array(rng, (300, 400), dtype), rand_array(rng, (9, 9), dtype)
    p = nc.get_fft_processor(dtype)
    for n in (32, 100, 250, 1024):
        a = rand_array(rng, (32, n), dtype)
        spec = p.forward(a)
        for _ in range(3):
            nc.conv_fft(x, k, nc.ConvMode.Same, nc.PaddingMode.Zeros)
            assert O.relerr(p.backward(spec), a)[0] <= (1e-5 if dtype == np.float32 else 1e-12)
    p.close()


# outer taps from kept spectra of x's tiles (fills of zero and repeating sides, x small) and
# transformed per tap (constant fills, x large): strides, dilation, views, several outer axes
@pytest.mark.parametrize("pm", ["zeros", "reflect", "circular", "replicate", ("const", 0.5)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64, np.complex128])
@pytest.mark.parametrize("shape,k,mode,dil", [((4, 40, 50), (3, 5, 7), "same", 1), ((9, 33, 31), (4, 3, 9), "full", 2),
                                              ((7, 60, 45), (3, 9, 5), ("custom", [3, 4, 2], [2, 3, 1]), 1),
                                              ((3, 4, 30, 41), (2, 3, 5, 6), "same", 1), ((16, 20, 20), (16, 3, 3), "valid", 1),
                                              ((40, 200, 260), (5, 3, 3), "same", 1)])
def test_outer_taps_kept_spectra(gpu, dtype, shape, k, mode, dil, pm):
    rng = np.random.default_rng(sum(shape) + sum(k))
    x = rand_array(rng, tuple(2 * n for n in shape), dtype)[tuple(slice(None, None, -2) for _ in shape)]
    try:
        check(x, rand_array(rng, k, dtype), mode, pm, dil)
    except O.OracleError:
        pytest.skip("refused by the reference")
