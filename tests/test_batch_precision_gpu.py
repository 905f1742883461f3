"""The autotuned batch that admits split BF16 products keeps FP32 for pairs
that FP32 computes at less cost, whatever the other pairs of the batch take."""
import numpy as np
import pytest

import ndconv as nc
from oracle import ndconv_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [40, 200, 400])
def test_short_signals_under_long_kernels_stay_fp32(gpu, count):
    """A matrix-core item makes 4096 outputs: for 600 it costs several times the
    one tile of 1024 points that FP32 takes.  The long signals beside them
    are better off in the queue.  Bar: 8 ulp of FP32 (a 1024-point transform's
    error is 1 to 2); BF16x3 sums of 512 products are off by 2^-18, 30 ulp."""
    rng = np.random.default_rng(count)
    n = np.array([600] * count + [60000] * 200)
    k = np.array([512] * count + [63] * 200)
    x = (rng.random(int(n.sum())) * 2 - 1).astype(np.float32)
    kv = (rng.random(int(k.sum())) * 2 - 1).astype(np.float32)
    import torch
    b = nc.BatchPlan(n, k, nc.ConvMode.Same, nc.PaddingMode.Zeros, algo="auto_bf16x3")
    y = b.run(torch.from_numpy(x).cuda(), torch.from_numpy(kv).cuda()).cpu().numpy()
    b.close()
    for i in range(count):
        ref = O.conv_fft(x[600 * i:600 * (i + 1)].astype(np.float64), kv[512 * i:512 * (i + 1)].astype(np.float64), "same",
                         "zeros")
        assert O.relerr(y[600 * i:600 * (i + 1)], ref)[0] <= 8 * 2.0 ** -23
