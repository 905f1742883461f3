"""Double-precision conv_fft by tiles against sums in 80 bits at random outputs:
no further off than the whole-array passes it replaced, whose errors (of the
outputs' norm) are the bars."""
import numpy as np
import pytest

import ndconv as nc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,mean,bar", [(1000003, 1023, 0.5, 1.80e-16), (1000003, 1023, 0.0, 5.03e-16),
                                          (60000, 255, 0.5, 1.93e-16), (60000, 255, 0.0, 4.20e-16),
                                          (5000, 31, 0.5, 2.47e-16), (5000, 31, 0.0, 3.94e-16)])
def test_rank1_error(gpu, n, k, mean, bar):
    rng = np.random.default_rng(0)
    x, kv = ((rng.random(s) if mean else rng.standard_normal(s)) for s in (n, k))
    got = nc.conv_fft(x, kv, nc.ConvMode.Same, nc.PaddingMode.Zeros)
    at = rng.integers(0, n, 3000)
    xp = np.pad(x, (k // 2, (k - 1) // 2)).astype(np.longdouble)
    ref = (xp[at[:, None] + np.arange(k)] * kv[::-1].astype(np.longdouble)).sum(1)
    assert np.sqrt(((got[at] - ref) ** 2).sum() / (ref ** 2).sum()) <= bar
