"""The batch's overlap-save tile runs at their edges: the longest kernels of
each tile class and the first ones past them, signals that end at, before and
after a tile, every border, pads longer than the signal, strides, dilation.
Against the FP64 oracle at 1e-5 normwise, the batch's bound for every form."""
import numpy as np
import pytest

from modes import conv_mode, padding_mode
from oracle import ndconv_oracle as O

import ndconv as nc

pytestmark = pytest.mark.gpu

TOL = 1e-5


def check(n, k, mode, pm, dil=1, rev=True, seed=0):
    rng = np.random.default_rng(seed)
    xs = [rng.uniform(-1, 1, a).astype(np.float32) for a in n]
    ks = [rng.uniform(-1, 1, b).astype(np.float32) for b in k]
    for algo in ("fft", "auto"):
        got = nc.conv_fft_batch(xs, ks, conv_mode(mode), padding_mode(pm), dil, rev, algo)
        for x, kv, g in zip(xs, ks, got):
            ref = O.conv_fft(x.astype(np.float64), kv.astype(np.float64), mode, pm, dil, rev)
            assert g.shape == ref.shape
            assert O.relerr(g, ref)[0] <= TOL, (algo, len(x), len(kv))


@pytest.mark.parametrize("points,k", [(1024, 1), (1024, 2), (1024, 31), (1024, 896), (4096, 897), (4096, 3584),
                                      (8192, 3585), (8192, 7168), (16384, 7169), (16384, 9000), (16384, 14337)])
def test_batch_tile_lengths(gpu, points, k):
    V = max(points - k + 1, 1)
    n = [1, V - 1 or 1, V, V + 1, 2 * V, 2 * V + 1, 5 * V + 7]
    check(n, [k] * len(n), "same", "zeros", seed=k)


@pytest.mark.parametrize("pm", ["zeros", "circular", "reflect", "replicate", ("const", -0.75)])
@pytest.mark.parametrize("mode", ["full", "same", ("custom", [40], [3])])
def test_batch_tile_borders(gpu, pm, mode):
    n, k = [77, 100, 1500, 9000, 31], [40, 1, 33, 60, 31]
    for dil, rev in ((1, True), (1, False), (3, True)):
        m = n if pm != "reflect" else [max(a, (b - 1) * dil + 41) for a, b in zip(n, k)]
        check(m, k, mode, pm, dil, rev, seed=dil)


@pytest.mark.parametrize("pm", ["circular", "replicate"])
def test_batch_tile_pads_longer_than_the_signal(gpu, pm):
    check([1, 3, 40, 500], [300, 64, 200, 1001], "same", pm, seed=9)
