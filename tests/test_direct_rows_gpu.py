"""The direct kernel's tile heights: 16 rows below one block a compute unit, 32
from there on, at sizes around both, for elements of 2 and 8 bytes that have
no matrix form of that rank.  Integers exactly, floats within the suite's bar."""
import numpy as np
import pytest

import ndconv as nc
from modes import conv_mode, padding_mode, rand_array
from oracle import ndconv_oracle as O

pytestmark = pytest.mark.gpu

BAR = {np.dtype(np.float64): 1e-12, np.dtype(np.complex64): 1e-5}


def check(x, k, mode, pm, dil):
    got = nc.conv(x, nc.with_dilation(k, dil), conv_mode(mode), padding_mode(pm))
    if x.dtype.kind in "iu":
        np.testing.assert_array_equal(got, O.conv(x, k, mode, pm, dil))
    else:
        ref = O.conv(x.astype(np.complex128 if x.dtype.kind == "c" else np.float64),
                     k.astype(np.complex128 if k.dtype.kind == "c" else np.float64), mode, pm, dil)
        assert got.shape == ref.shape
        assert O.relerr(got, ref)[0] <= BAR[x.dtype]


@pytest.mark.parametrize("dtype", [np.float64, np.complex64, np.int64])
@pytest.mark.parametrize("shape", [(1, 63), (15, 64), (16, 65), (17, 128), (33, 200), (479, 1024), (480, 1025), (513, 1088)])
def test_rows(gpu, dtype, shape):
    rng = np.random.default_rng(shape[0] + shape[1])
    check(rand_array(rng, shape, dtype), rand_array(rng, (3, 5), dtype), "same", "zeros", 1)
    check(rand_array(rng, shape, dtype), rand_array(rng, (1, 9), dtype), ("custom", [2, 5], [2, 2]), "replicate", 2)


@pytest.mark.parametrize("dtype", [np.float32, np.int16, np.int64])
def test_rows_rank3(gpu, dtype):
    rng = np.random.default_rng(7)
    x = rand_array(rng, (5, 37, 70), dtype)
    k = rand_array(rng, (2, 3, 5), dtype)
    if np.dtype(dtype) == np.float32:
        got = nc.conv(x, k, conv_mode("full"), padding_mode("zeros"))
        assert O.relerr(got, O.conv(x.astype(np.float64), k.astype(np.float64), "full", "zeros", 1))[0] <= 1e-5
    else:
        check(x, k, "full", "zeros", 1)
