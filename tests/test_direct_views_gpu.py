"""Direct convolution of large views reversed along an outer axis: the planes
of such a view start below its first element, and padding cells are still not
read from the array."""
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
