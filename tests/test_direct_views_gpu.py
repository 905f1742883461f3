"""Direct convolution away from the usual plans: large views reversed along an
outer axis, whose planes start below the first element (padding cells are
still not read from the array), and dilations of 0 or past every offset."""
import numpy as np
import pytest

import ndconv as nc
from modes import conv_mode, padding_mode
from oracle import ndconv_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pm", ["zeros", ("custom", ["zeros", ("const", 3), "zeros"])])
def test_reversed_planes_of_600_mib(gpu, pm):
    rng = np.random.default_rng(3)
    x = np.tile(rng.integers(1, 100, (1, 1024, 1024), dtype=np.int8), (600, 1, 1))
    x += np.arange(600, dtype=np.int8)[:, None, None] % 5
    k = rng.integers(-9, 9, (1, 3, 3), dtype=np.int8)
    mode = ("explicit", [[0, 0], [1, 1], [1, 1]], [100, 1, 1])
    got = nc.conv(x[::-1], k, conv_mode(mode), padding_mode(pm))
    np.testing.assert_array_equal(got, O.conv(x[::-1][::100], k, ("explicit", mode[1], [1, 1, 1]), pm))


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32, np.int8])
@pytest.mark.parametrize("shape,ks,dil", [((90,), (3,), 0), ((40, 270), (3, 4), [0, 1]), ((40, 270), (3, 4), [2, 0]),
                                          ((40, 270), (1, 4), [1 << 50, 1]), ((4, 20, 30), (2, 3, 2), [0, 1, 0])])
def test_any_dilation(gpu, dtype, shape, ks, dil):
    """Dilation 0 (every tap meets the same sample) and any dilation of one tap."""
    rng = np.random.default_rng(4)
    x, k = rng.integers(-9, 10, shape).astype(dtype), rng.integers(-9, 10, ks).astype(dtype)
    got = nc.conv(x, nc.with_dilation(k, dil), conv_mode("same"), padding_mode("replicate"))
    np.testing.assert_array_equal(got, O.conv(x, k, "same", "replicate", dil))   # whole numbers: exact in every type


def test_stride_that_fills_lds(gpu):
    """The region of 16 rows at stride 10 leaves no room for the offset tables."""
    rng = np.random.default_rng(5)
    x, k = (rng.integers(-9, 10, s) + 1j * rng.integers(-9, 10, s) for s in ((20, 700), (3, 3)))
    mode = ("explicit", [[1, 1], [1, 1]], [1, 10])
    got = nc.conv(x.astype(np.complex128), k.astype(np.complex128), conv_mode(mode), padding_mode("circular"))
    np.testing.assert_array_equal(got, O.conv(x, k, mode, "circular"))
