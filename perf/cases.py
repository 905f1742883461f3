"""The calls whose speed is measured: convolutions through the package's public entry points.

A case is a dict of plain values:

    op       "conv_fft", "baked" (conv_fft with a kept kernel spectrum), "conv", "conv_bf16x3",
             "processor" (FftProcessor forward, then backward) or "batch" (BatchPlan.run)
    dtype    element type
    shape, kernel    sizes, axes separated by "x" (single problems)
    mode, border, dilation, stride, reverse    the options of the call (a stride other than 1 is a
             ConvMode.Explicit with the mode's padding; a border may name one type per axis)
    count, n_min, n_max, k_min, k_max, lens, algo    an uneven batch: its lengths are log-uniform,
             from `lens`

`run` makes one pass; `exact` is the same result from plain torch in 64 bits.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ndarray-conv_amd"))

import ndconv as nc  # noqa: E402

DEVICE = "cuda:0"
CONST = 0.5   # the pad value of a "const" border


def _case(op, dtype, **kw):
    c = {"op": op, "dtype": dtype}
    if op == "batch":
        c.update(count=1, n_min=256, n_max=262144, k_min=3, k_max=1023, lens=5, algo="auto")
    c.update(mode="same", border="zeros", dilation=1, stride=1, reverse=True)
    c.update(kw)
    return c


def listed():
    return [
        # One short signal filtered once: the smallest call, where latency and launches count.
        _case("conv_fft", "float32", name="fft_1d_5000_f32", shape="5000", kernel="31"),
        # A small picture smoothed with a small filter in the crate's default float type.
        _case("conv", "float64", name="conv_480x640_k5x5_f64", shape="480x640", kernel="5x5", border="reflect"),
        # An ordinary two-dimensional FFT convolution, a border type per axis, dilated.
        _case("conv_fft", "float32", name="fft_200x5000_f32", shape="200x5000", kernel="11x31", dilation=2,
              border="reflect,circular"),
        # A complex volume (a field sampled on a small grid), full output.
        _case("conv_fft", "complex64", name="fft_10x100x200_c64", shape="10x100x200", kernel="5x11x31", mode="full"),
        # Whole numbers, bit-exact: quantised samples with a medium filter.
        _case("conv", "int32", name="conv_200x5000_i32", shape="200x5000", kernel="11x31", border="reflect,circular"),
        # A large picture, a large filter, decimated on the way, exact FP32.
        _case("conv", "float32", name="conv_4096x4096_f32", shape="4096x4096", kernel="31x31", mode="valid",
              border="replicate", dilation=2, stride=2),
        # The same with split BF16 on the matrix cores.
        _case("conv_bf16x3", "float32", name="conv_4096x4096_bf16x3", shape="4096x4096", kernel="31x31", mode="valid",
              border="replicate", dilation=2, stride=2),
        # A very large picture (512 MiB in and out) by FFT.
        _case("conv_fft", "float32", name="fft_4096x32768_f32", shape="4096x32768", kernel="11x31", dilation=2,
              border="reflect,circular"),
        # A long double-precision recording, ragged length, passed through one long kept filter.
        _case("baked", "float64", name="baked_1000003_f64", shape="1000003", kernel="1023", border="reflect"),
        # The transforms by themselves, as a spectral program uses them.
        _case("processor", "float32", name="processor_256x5120_f32", shape="256x5120"),
        # A few hundred recordings of very different lengths, FP32 only (the default algorithm).
        _case("batch", "float32", name="batch_509_f32", count=509, n_max=65536, k_max=255, lens=11, border="reflect"),
        # Thousands of them, matrix cores admitted.
        _case("batch", "float32", name="batch_4096_bf16x3", count=4096, n_min=512, border="circular",
              algo="auto_bf16x3"),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    border = rng.choice(["zeros", "const", "reflect", "replicate", "circular"])
    mode = rng.choice(["same", "same", "full", "valid"])
    kw = {"border": border, "mode": mode, "reverse": rng.random() < 0.8}
    op = rng.choice(["fft1", "fft2", "fft2", "fft3", "conv", "conv", "bf16x3", "processor", "batch", "batch"])
    if op == "fft1":
        n = _log(rng, 2100, 1 << 20)
        return _case(rng.choice(["conv_fft", "conv_fft", "baked"]), rng.choice(["float32", "float32", "float64", "complex64"]),
                     shape="%d" % n, kernel="%d" % _log(rng, 3, 1023), dilation=rng.choice([1, 1, 2]), **kw)
    if op == "fft2":
        h, w = _log(rng, 100, 4096), _log(rng, 100, 8192)
        return _case(rng.choice(["conv_fft", "conv_fft", "conv_fft", "baked"]), rng.choice(["float32", "float32", "float64"]),
                     shape="%dx%d" % (h, w), kernel="%dx%d" % (_log(rng, 3, 31), _log(rng, 3, 31)),
                     dilation=rng.choice([1, 1, 2, 3]), stride=rng.choice([1, 1, 1, 2]), **kw)
    if op == "fft3":
        return _case("conv_fft", rng.choice(["float32", "complex64"]),
                     shape="%dx%dx%d" % (_log(rng, 10, 64), _log(rng, 40, 200), _log(rng, 40, 400)),
                     kernel="%dx%dx%d" % (rng.randint(2, 7), rng.randint(3, 11), rng.randint(3, 31)), **kw)
    if op == "conv":
        h, w = _log(rng, 64, 2048), _log(rng, 64, 4096)
        return _case("conv", rng.choice(["float32", "float32", "float64", "int32", "int16"]), shape="%dx%d" % (h, w),
                     kernel="%dx%d" % (_log(rng, 3, 15), _log(rng, 3, 31)), dilation=rng.choice([1, 1, 2]),
                     stride=rng.choice([1, 1, 2]), **kw)
    if op == "bf16x3":
        s, d = rng.choice([(1, 1), (1, 2), (2, 2)])
        return _case("conv_bf16x3", "float32", shape="%dx%d" % (_log(rng, 256, 4096), _log(rng, 256, 4096)),
                     kernel="%dx%d" % (_log(rng, 7, 31), _log(rng, 7, 31)), dilation=d, stride=s, **kw)
    if op == "processor":
        return _case("processor", rng.choice(["float32", "float32", "float64", "complex64"]),
                     shape="%dx%d" % (2 * _log(rng, 16, 256) * rng.choice([1, 3]), 2 * _log(rng, 64, 2560)))
    k_max, mode = _log(rng, 31, 1023), rng.choice(["same", "same", "full"])
    n_min = max(256, k_max if mode == "full" else k_max // 2 + 1)   # no pad reaches past its signal
    return _case("batch", "float32", count=_log(rng, 32, 2048), n_min=n_min, n_max=_log(rng, 4096, 262144), k_max=k_max,
                 lens=rng.randint(1, 1 << 20), border=border, mode=mode, reverse=kw["reverse"],
                 algo=rng.choice(["auto", "auto", "auto_bf16x3"]))


# What a case means ---------------------------------------------------------

def _dims(text):
    return [int(v) for v in text.split("x")]


def _borders(c, rank):
    b = c["border"].split(",")
    return b if len(b) == rank else b * rank


def _pads(c, kernel):
    """The (front, back) padding of each axis."""
    out = []
    for k in kernel:
        kd = (k - 1) * c["dilation"] + 1
        if c["mode"] == "full":
            out.append((kd - 1, kd - 1))
        elif c["mode"] == "same":
            out.append((kd // 2, (kd - 1) // 2))
        else:
            out.append((0, 0))
    return out


def _conv_mode(c, kernel):
    if c["stride"] != 1:
        return nc.ConvMode.Explicit([list(p) for p in _pads(c, kernel)], [c["stride"]] * len(kernel))
    return {"full": nc.ConvMode.Full, "same": nc.ConvMode.Same, "valid": nc.ConvMode.Valid}[c["mode"]]


def _padding_mode(c, rank):
    plain = {"zeros": nc.PaddingMode.Zeros, "reflect": nc.PaddingMode.Reflect, "replicate": nc.PaddingMode.Replicate,
             "circular": nc.PaddingMode.Circular}
    names = c["border"].split(",")
    if len(names) == 1:
        return nc.PaddingMode.Const(CONST) if names[0] == "const" and c["dtype"][:3] != "int" else \
            nc.PaddingMode.Const(1) if names[0] == "const" else plain[names[0]]
    return nc.PaddingMode.Custom([getattr(nc.BorderType, n.capitalize()) for n in names])


def _lens(c):
    """Signal and kernel lengths of an uneven batch, log-uniform."""
    rng = np.random.default_rng(c["lens"])
    pick = lambda lo, hi: np.clip(np.floor(np.exp(rng.uniform(np.log(lo), np.log(hi + 1), c["count"]))), lo,
                                  hi).astype(np.int64)
    return pick(c["n_min"], c["n_max"]), pick(c["k_min"], c["k_max"])


def _inputs(c, seed):
    """Data and taps on the GPU, from the seed alone."""
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    dt = getattr(torch, c["dtype"])
    if c["op"] == "batch":
        n, k = _lens(c)
        return [torch.rand(int(s.sum()), generator=g, device=DEVICE) * 2 - 1 for s in (n, k)]
    shapes = [_dims(c["shape"])] + ([_dims(c["kernel"])] if "kernel" in c else [])
    if dt in (torch.int32, torch.int16):
        return [torch.randint(-8, 9, s, generator=g, device=DEVICE, dtype=dt) for s in shapes]
    if c["op"] in ("conv_fft", "baked") and not dt.is_complex:   # sample values in [0, 1)
        return [torch.rand(s, generator=g, device=DEVICE, dtype=dt) for s in shapes]
    return [torch.randn(s, generator=g, device=DEVICE, dtype=dt) for s in shapes]


def prepare(case, seed):
    c = case
    ins = _inputs(c, seed)
    state = {"case": c, "x": ins[0]}
    if c["op"] == "processor":
        state["processor"] = nc.get_fft_processor(np.dtype(c["dtype"]))
        return state
    if c["op"] == "batch":
        n, k = _lens(c)
        mode = {"full": nc.ConvMode.Full, "same": nc.ConvMode.Same}[c["mode"]]
        state["k"] = ins[1]
        state["plan"] = nc.BatchPlan(n, k, mode, _padding_mode(c, 1), c["dilation"], c["reverse"], algo=c["algo"])
        return state
    kernel = _dims(c["kernel"])
    k = nc.with_dilation(ins[1], c["dilation"])
    state["k"] = k if c["reverse"] else k.no_reverse()
    state["mode"], state["pad"] = _conv_mode(c, kernel), _padding_mode(c, len(kernel))
    if c["op"] == "baked":
        state["baked"] = nc.conv_fft_bake(state["x"], state["k"], state["mode"], state["pad"])
    return state


def run(state):
    op = state["case"]["op"]
    if op == "conv_fft":
        return nc.conv_fft(state["x"], state["k"], state["mode"], state["pad"])
    if op == "baked":
        return nc.conv_fft_with_baked(state["x"], state["baked"])
    if op == "conv":
        return nc.conv(state["x"], state["k"], state["mode"], state["pad"])
    if op == "conv_bf16x3":
        return nc.conv(state["x"], state["k"], state["mode"], state["pad"], algo="bf16x3")
    if op == "batch":
        return state["plan"].run(state["x"], state["k"])
    spectrum = state["processor"].forward(state["x"])
    return spectrum, state["processor"].backward(spectrum)


def _out_len(n, k, pads, c):
    return (n + pads[0] + pads[1] - (k - 1) * c["dilation"] - 1) // c["stride"] + 1


def work(case):
    c = case
    e = torch.empty(0, dtype=getattr(torch, c["dtype"])).element_size()
    mul = 4 if c["dtype"].startswith("complex") else 1   # real operations a product and sum stand for
    if c["op"] == "processor":
        n = math.prod(_dims(c["shape"]))
        spec = n * (8 if c["dtype"] in ("float32", "complex64") else 16) // (1 if mul == 4 else 2)
        return {"bytes": 2 * (n * e + spec), "flops": 2 * 2.5 * n * math.log2(n) * (2 if mul == 4 else 1)}
    if c["op"] == "batch":
        n, k = _lens(c)
        out = n + (k - 1) if c["mode"] == "full" else n
        fft = 2 * 2.5 * (n + k) * np.log2(n + k)
        return {"bytes": int(4 * (n.sum() + k.sum() + out.sum())), "flops": float(np.minimum(fft, 2.0 * out * k).sum())}
    shape, kernel = _dims(c["shape"]), _dims(c["kernel"])
    outs = math.prod(_out_len(n, k, p, c) for n, k, p in zip(shape, kernel, _pads(c, kernel)))
    n, taps = math.prod(shape), math.prod(kernel)
    flops = 2.0 * outs * taps * mul
    if c["op"] in ("conv_fft", "baked"):
        flops = min(flops, 2 * 2.5 * n * math.log2(n) * (2 if mul == 4 else 1))
    return {"bytes": e * (n + taps + outs), "flops": flops}


# The same results from torch in 64 bits -------------------------------------

def _pad_index(n, front, back, border):
    """Where each position of a padded axis reads (-1: the pad value)."""
    i = torch.arange(-front, n + back, device=DEVICE)
    if border in ("zeros", "const"):
        return torch.where((i < 0) | (i >= n), -1, i)
    if border == "replicate":
        return i.clamp(0, n - 1)
    if border == "circular":
        return i % n
    i = i.abs()
    return torch.where(i >= n, 2 * (n - 1) - i, i)


def _pow2(n):
    return 1 << max(0, (n - 1).bit_length())


def _linear(x, k, pads, borders, const, c):
    """Padded, dilated, strided convolution (or correlation) by a 64-bit FFT."""
    rank = x.dim()
    wide = torch.complex128 if x.is_complex() else torch.float64
    x, k = x.to(wide), k.to(wide)
    for a in range(rank):
        idx = _pad_index(x.shape[a], pads[a][0], pads[a][1], borders[a])
        y = x.index_select(a, idx.clamp(min=0))
        if borders[a] in ("zeros", "const"):
            out = (idx < 0).reshape([-1 if b == a else 1 for b in range(rank)])
            y = y.masked_fill(out, const if borders[a] == "const" else 0.0)
        x = y
    if not c["reverse"]:
        k = k.flip(list(range(rank)))
    d = c["dilation"]
    kd = k.new_zeros([(s - 1) * d + 1 for s in k.shape])
    kd[tuple(slice(None, None, d) for _ in range(rank))] = k
    size = [_pow2(s) for s in x.shape]
    axes = list(range(rank))
    if x.is_complex():
        y = torch.fft.fftn(x, size, axes).mul_(torch.fft.fftn(kd, size, axes))
        y = torch.fft.ifftn(y, size, axes)
    else:
        y = torch.fft.rfftn(x, size, axes).mul_(torch.fft.rfftn(kd, size, axes))
        y = torch.fft.irfftn(y, size, axes)
    return y[tuple(slice(kk - 1, s, c["stride"]) for kk, s in zip(kd.shape, x.shape))].contiguous()


def exact(case, seed):
    c = case
    ins = _inputs(c, seed)
    if c["op"] == "processor":
        x = ins[0]
        wide = x.to(torch.complex128 if x.is_complex() else torch.float64).cpu().numpy()
        axes = tuple(range(wide.ndim))
        spec = np.fft.fftn(wide, axes=axes) if x.is_complex() else np.fft.rfftn(wide, axes=axes)
        return np.ascontiguousarray(np.moveaxis(spec, 0, -1)), wide
    if c["op"] == "batch":
        n, k = _lens(c)
        xo, ko = np.concatenate([[0], np.cumsum(n)]), np.concatenate([[0], np.cumsum(k)])
        out = []
        for i in range(len(n)):
            x, kv = ins[0][xo[i]:xo[i + 1]], ins[1][ko[i]:ko[i + 1]]
            out.append(_linear(x, kv, _pads(c, [int(k[i])]), _borders(c, 1), CONST, c))
        return torch.cat(out)
    x, k = ins
    const = CONST if c["dtype"][:3] != "int" else 1
    y = _linear(x, k, _pads(c, _dims(c["kernel"])), _borders(c, x.dim()), const, c)
    return y.round().to(x.dtype) if c["dtype"][:3] == "int" else y
