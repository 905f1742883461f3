"""Host side of a call: the closed-form check of the border fills against the
map that replays them, and the keys under which prepared calls are kept."""
import numpy as np
import pytest

import ndconv as nc

B, P, M = nc.BorderType, nc.PaddingMode, nc.ConvMode


@pytest.mark.parametrize("fft", [False, True])
@pytest.mark.parametrize("n", range(1, 9))
def test_fill_check_agrees_with_the_map(n, fft):
    """plan() checks in closed form what border_map() finds by replaying."""
    for front in (B.Reflect, B.Circular, B.Zeros):
        for back in (B.Reflect, B.Replicate):
            for p0 in range(14):
                for p1 in range(14):
                    mode, pm = M.Explicit([[p0, p1]], [1]), P.Explicit([[front, back]])
                    got = []
                    for call in (lambda: nc.plan((n,), (1,), mode, pm, fft=fft),
                                 lambda: nc.border_map((n,), (1,), mode, pm, 0, fft=fft)):
                        try:
                            call()
                            got.append(None)
                        except nc.Error as e:
                            got.append(type(e))
                    assert got[0] is got[1], (front, back, p0, p1, got)


def test_call_keys_tell_values_apart():
    pads = [P.Zeros, P.Reflect, P.Const(0.0), P.Const(-0.0), P.Const(1), P.Const(1.0), P.Const(True),
            P.Const(float("nan")), P.Const(0.1), P.Const(np.float32(0.1)), P.Const(np.float64(0.1)), P.Const(1 + 0j),
            P.Custom([B.Zeros]), P.Custom([B.Const(2.0)]), P.Custom([B.Const(2)]),
            P.Explicit([[B.Zeros, B.Const(2.0)]]), P.Explicit([[B.Const(2.0), B.Zeros]])]
    keys = [nc._pad_key(p) for p in pads]
    assert len(set(keys)) == len(keys)
    modes = [M.Full, M.Same, M.Valid, M.Custom([1], [1]), M.Custom([1], [2]), M.Explicit([[1, 1]], [1]),
             M.Explicit([[1, 2]], [1])]
    assert len({nc._mode_key(m) for m in modes}) == len(modes)
    with pytest.raises(TypeError):   # contents unknown: never kept
        nc._pad_key(P.Const(np.array(0.5)))


@pytest.mark.parametrize("border", ["Zeros", "Reflect", "Replicate", "Circular"])
def test_unread_planes_are_looked_over(border):
    """conv_fft by tiles that are transformed per tap (x past 8 MB of spectra)
    adds the look for non-finite values, a launch of no LDS beside the fix-up's,
    where some plane of x meets no tap."""
    bt = getattr(B, border)
    for n, k, d, s, p0, p1 in [(n, k, d, s, p0, p1) for n in (24, 25, 31) for k in (1, 2, 3) for d in (1, 2, 5, 13)
                               for s in (1, 2, 3, 7) for p0 in (0, 1, 4) for p1 in (0, 3)]:
        if n + p0 + p1 < (k - 1) * d + 1:
            continue
        pm = P.Custom([bt, B.Zeros, B.Zeros])
        mode = M.Explicit([[p0, p1], [0, 0], [0, 0]], [s, 1, 1])
        out = nc.plan((n, 300, 260), (k, 3, 3), mode, pm, dilation=[d, 1, 1], fft=True)["out_shape"][0]
        read = {o * s + t * d - p0 for o in range(out) for t in range(k)}
        got = nc.fft_launch_plan((n, 300, 260), (k, 3, 3), mode, pm, dilation=[d, 1, 1])
        if not set(range(n)) <= read:
            assert len([g for g in got if g[0] == 0]) == 2, (n, k, d, s, p0, p1, got)
