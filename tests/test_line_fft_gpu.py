"""The processor's line transforms at the lengths where their form changes: one
stage, a radix without a butterfly, odd real lines, two and more stages, lines
of several radices; blocks of 1 to 16 columns with a partial last one."""
import numpy as np
import pytest

from oracle import ndconv_oracle as O

import ndconv as nc

pytestmark = pytest.mark.gpu

# one rounding an operation: log2 of the points times a few units in the last place
EPS = {np.float32: 2.0 ** -24, np.float64: 2.0 ** -53}


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("real", [np.float32, np.float64])
@pytest.mark.parametrize("rows,cols", [(1, 2), (1, 16), (3, 7), (2, 32), (5, 11), (16, 33), (17, 24), (32, 30), (48, 96),
                                       (60, 200), (256, 40), (121, 256), (100, 1000), (512, 6), (7, 5120), (33, 2 * 169)])
def test_processor_line_forms(gpu, rows, cols, real, cplx):
    rng = np.random.default_rng(rows * 10000 + cols)
    x = rng.uniform(-1, 1, (rows, cols)).astype(real)
    if cplx:
        x = x + 1j * rng.uniform(-1, 1, (rows, cols)).astype(real)
    ctype = np.complex64 if real is np.float32 else np.complex128
    x = x.astype(ctype) if cplx else x
    p = nc.get_fft_processor(x.dtype.type)
    spec = p.forward(x)
    want = O.processor_forward(x.astype(np.complex128 if cplx else np.float64))
    tol = 8 * np.log2(rows * cols + 1) * EPS[real]
    got = np.asarray(spec)
    assert got.shape == want.shape
    assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
    back = p.backward(spec)
    assert np.linalg.norm(back - x) <= 2 * tol * np.linalg.norm(x)
