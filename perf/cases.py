"""Performance cases: the transforms and convolutions that users of kfr_amd run, over their real ranges.

listed() names the cases, draw() makes further ones from the same ranges, prepare() builds what a
program holds before the call (inputs, outputs, the plan), run() is one pass through the public API,
work() the bytes and operations that a pass cannot do without, and exact() the same results in FP64 by
torch or numpy.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import kfr_amd
from kfr_amd.autograd import fft_convolve

REAL = {"f32": torch.float32, "f64": torch.float64}
COMPLEX = {"f32": torch.complex64, "f64": torch.complex128}
NP_REAL = {"f32": np.float32, "f64": np.float64}
NP_COMPLEX = {"f32": np.complex64, "f64": np.complex128}
HALF = {"bf16": torch.bfloat16, "f16": torch.float16}


def listed():
    return [
        # one frame of a running program, transformed as it arrives: the call and launch cost
        {"name": "c2c_f32_1024_one", "kind": "c2c", "n": 1024, "batch": 1, "dtype": "f32", "direction": "forward"},
        # the benchmark's round trip: forward and inverse of a small batch
        {"name": "c2c_f32_4096x256_both", "kind": "c2c", "n": 4096, "batch": 256, "dtype": "f32", "direction": "both"},
        # 20 ms frames at 48 kHz, a recording's worth: a length that is no power of two
        {"name": "c2c_f32_960x16384", "kind": "c2c", "n": 960, "batch": 16384, "dtype": "f32", "direction": "forward"},
        # double precision, an odd mixed length beyond one workgroup (in the parity tests)
        {"name": "c2c_f64_30240x256_inv", "kind": "c2c", "n": 30240, "batch": 256, "dtype": "f64",
         "direction": "inverse"},
        # the long end of the benchmark's sweep, 1 GiB of input
        {"name": "c2c_f32_4Mx32", "kind": "c2c", "n": 1 << 22, "batch": 32, "dtype": "f32", "direction": "forward"},
        # the benchmark's long real signals (2^14 * 3 * 5^4 points), spectrum and back
        {"name": "real_f32_30720000x8_both", "kind": "real", "n": 30720000, "batch": 8, "dtype": "f32"},
        # the benchmark's DCT-II, and DCT-III back
        {"name": "dct_f32_65536x1024_both", "kind": "dct", "n": 65536, "batch": 1024, "dtype": "f32"},
        # a training step through the benchmark's convolution: output and both gradients
        {"name": "conv_f32_1Mx128_grad", "kind": "conv", "n": 1 << 20, "taps": 4095, "batch": 128, "dtype": "f32",
         "shared": False},
        # the benchmark's uneven batch: every 7-smooth length in [18, 8192] and the primes in [17, 127]
        {"name": "uneven_f32_20000", "kind": "uneven", "count": 20000, "most": 8192, "dtype": "f32", "lengths": 3},
        # half-precision storage, the benchmark's size
        {"name": "half_bf16_1Mx64", "kind": "half", "n": 1 << 20, "batch": 64, "dtype": "bf16",
         "direction": "forward"},
        # the spectrum of one image and back
        {"name": "image_f32_1080x1920_both", "kind": "md_real", "d0": 1080, "d1": 1920, "d2": 0, "dtype": "f32"},
        # a streaming filter fed block by block
        {"name": "filter_f32_4095_1024x64", "kind": "filter", "taps": 4095, "block": 1024, "calls": 64,
         "dtype": "f32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """A power of two, a 7-smooth length up to 2^20 or any length up to 2^16, spread over the logarithm
    of the range."""
    pick = rng.random()
    if pick < 0.35:
        return min(hi, 1 << max(1, int(round(math.log2(_log_int(rng, lo, hi))))))
    if pick < 0.8:
        n = _log_int(rng, lo, min(hi, 1 << 20))
        while not _smooth(n):
            n -= 1
        return max(2, n)
    return _log_int(rng, lo, min(hi, 1 << 16))


def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def _batch(rng, n, total):
    return max(1, min(total // n, _log_int(rng, 1, max(1, total // n) + 1)))


def draw(rng):
    kind = rng.choice(["c2c", "c2c", "c2c", "c2c", "real", "real", "dct", "conv", "uneven", "half", "md", "filter"])
    dtype = rng.choice(["f32", "f32", "f64"])
    total = 1 << 24
    if kind == "c2c":
        n = _length(rng, 16, 1 << 22)
        return {"kind": kind, "n": n, "batch": _batch(rng, n, total), "dtype": dtype,
                "direction": rng.choice(["forward", "inverse", "both"])}
    if kind == "real":
        n = 2 * _length(rng, 16, 1 << 22)
        return {"kind": kind, "n": n, "batch": _batch(rng, n, total), "dtype": dtype}
    if kind == "dct":
        n = _length(rng, 16, 1 << 18)
        return {"kind": kind, "n": n, "batch": _batch(rng, n, total), "dtype": dtype}
    if kind == "conv":
        taps = _log_int(rng, 15, 4095)
        n = _log_int(rng, 4 * taps, 1 << 20)
        return {"kind": kind, "n": n, "taps": taps, "batch": _batch(rng, n, total), "dtype": dtype,
                "shared": rng.random() < 0.5}
    if kind == "uneven":
        return {"kind": kind, "count": _log_int(rng, 100, 8000), "most": rng.choice([512, 2048, 4096]),
                "dtype": dtype, "lengths": rng.randrange(1 << 20)}
    if kind == "half":
        n = 1 << rng.randint(5, 22)
        return {"kind": kind, "n": n, "batch": _batch(rng, n, total), "dtype": rng.choice(["bf16", "f16"]),
                "direction": rng.choice(["forward", "inverse"])}
    if kind == "md":
        if rng.random() < 0.5:
            shape = (_length(rng, 16, 2048), _length(rng, 16, 2048), 0)
        else:
            shape = tuple(_length(rng, 8, 160) for _ in range(3))
        kind = rng.choice(["md", "md_real"])
        d0, d1, d2 = shape
        if kind == "md_real":  # the real axis is the last one, of even length
            d1, d2 = (2 * ((d1 + 1) // 2), 0) if d2 == 0 else (d1, 2 * ((d2 + 1) // 2))
        return {"kind": kind, "d0": d0, "d1": d1, "d2": d2, "dtype": dtype}
    return {"kind": "filter", "taps": _log_int(rng, 16, 8191), "block": 1 << rng.randint(7, 12),
            "calls": rng.randint(4, 48), "dtype": dtype}


def _shape(case):
    return tuple(d for d in (case["d0"], case["d1"], case["d2"]) if d)


def _lengths(case):
    """Lengths and directions of an uneven batch (the batch's own layout, the same for every input)."""
    smooth = {2 ** a * 3 ** b * 5 ** c * 7 ** d for a in range(14) for b in range(9) for c in range(6)
              for d in range(5)}
    primes = [p for p in range(17, 128) if all(p % q for q in range(2, int(p ** 0.5) + 1))]
    table = np.array(sorted({v for v in smooth if 18 <= v <= case["most"]} | set(primes)), dtype=np.int64)
    rng = np.random.default_rng(case["lengths"])
    return rng.choice(table, case["count"]), rng.integers(0, 2, case["count"]).astype(np.int32)


def _taps(count, dtype, gen):
    """Hann-windowed sinc low-pass (cutoff 0.2 of the sampling rate) plus a little noise, (rows, taps)."""
    rows, taps = count
    k = torch.arange(taps, dtype=torch.float64, device="cuda") - (taps - 1) / 2
    h = 0.4 * torch.sinc(0.4 * k) * torch.hann_window(taps, periodic=False, dtype=torch.float64, device="cuda")
    noise = torch.randn(rows, taps, dtype=torch.float64, device="cuda", generator=gen)
    return (h + 1e-3 * noise).to(REAL[dtype])


def _inputs(case, seed):
    """The input tensors of a pass, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, dt = case["kind"], case["dtype"]

    def normal(*shape):
        return torch.randn(*shape, dtype=REAL[dt], device="cuda", generator=gen)

    if kind == "c2c":
        return {"x": torch.view_as_complex(normal(case["batch"], case["n"], 2))}
    if kind in ("real", "dct"):
        return {"x": normal(case["batch"], case["n"])}
    if kind == "conv":
        taps = _taps((1 if case["shared"] else case["batch"], case["taps"]), dt, gen)
        return {"x": normal(case["batch"], case["n"]), "h": taps[0].clone() if case["shared"] else taps,
                "g": normal(case["batch"], case["n"] + case["taps"] - 1)}
    if kind == "uneven":
        total = int(_lengths(case)[0].sum())
        u = torch.rand(total, 2, dtype=REAL[dt], device="cuda", generator=gen)
        return {"x": torch.view_as_complex(u * 2 - 1)}
    if kind == "half":
        u = torch.randn(case["batch"], case["n"], 2, device="cuda", generator=gen)
        return {"x": (u * math.sqrt(0.5)).to(HALF[dt])}
    if kind == "md":
        return {"x": torch.view_as_complex(normal(*_shape(case), 2))}
    if kind == "md_real":
        return {"x": normal(*_shape(case))}
    h = _taps((1, case["taps"]), dt, gen)[0]
    return {"x": normal(case["calls"], case["block"]), "h": h}


def prepare(case, seed):
    s = _inputs(case, seed)
    kind, dt = case["kind"], case["dtype"]
    s["case"] = case
    if kind == "c2c":
        s["plan"] = kfr_amd.dft_plan(case["n"], NP_COMPLEX[dt])
        s["y"] = torch.empty_like(s["x"])
        if case["direction"] == "both":
            s["z"] = torch.empty_like(s["x"])
    elif kind == "real":
        s["plan"] = kfr_amd.dft_plan_real(case["n"], kfr_amd.CCs, NP_REAL[dt])
        s["y"] = torch.empty(case["batch"], case["n"] // 2 + 1, dtype=COMPLEX[dt], device="cuda")
        s["z"] = torch.empty_like(s["x"])
    elif kind == "dct":
        s["plan"] = kfr_amd.dct_plan(case["n"], NP_REAL[dt])
        s["y"], s["z"] = torch.empty_like(s["x"]), torch.empty_like(s["x"])
    elif kind == "conv":
        s["x"].requires_grad_()
        s["h"].requires_grad_()
    elif kind == "uneven":
        sizes, inverse = _lengths(case)
        s["plan"] = kfr_amd.dft_batch(sizes, inverse, NP_COMPLEX[dt])
        s["y"] = torch.empty_like(s["x"])
    elif kind == "half":
        s["plan"] = kfr_amd.dft_plan_half(case["n"], dt)
        s["y"] = torch.empty_like(s["x"])
    elif kind == "md":
        s["plan"] = kfr_amd.dft_plan_md(_shape(case), NP_COMPLEX[dt])
        s["y"] = torch.empty_like(s["x"])
    elif kind == "md_real":
        s["plan"] = kfr_amd.dft_plan_md_real(_shape(case), False, NP_REAL[dt])
        s["y"] = torch.empty(s["plan"].complex_size(), dtype=COMPLEX[dt], device="cuda")
        s["z"] = torch.empty_like(s["x"])
        s["temp"] = torch.empty(max(1, s["plan"].temp_size), dtype=torch.uint8, device="cuda")
    else:
        s["plan"] = kfr_amd.convolve_filter(s["h"].cpu().numpy(), case["block"])
        s["y"] = torch.empty_like(s["x"])
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "c2c":
        if case["direction"] == "both":
            s["plan"].execute_batch(s["y"], s["x"], case["batch"])
            s["plan"].execute_batch(s["z"], s["y"], case["batch"], inverse=True)
            return s["y"], s["z"]
        return s["plan"].execute_batch(s["y"], s["x"], case["batch"], inverse=case["direction"] == "inverse")
    if kind in ("real", "dct"):
        s["plan"].execute_batch(s["y"], s["x"], case["batch"])
        s["plan"].execute_batch(s["z"], s["y"], case["batch"], inverse=True)
        return s["y"], s["z"]
    if kind == "conv":
        y = fft_convolve(s["x"], s["h"])
        dx, dh = torch.autograd.grad(y, (s["x"], s["h"]), s["g"])
        return y.detach(), dx, dh
    if kind == "uneven":
        return s["plan"].execute(s["y"], s["x"])
    if kind == "half":
        return s["plan"].execute_batch(s["y"], s["x"], case["batch"], inverse=case["direction"] == "inverse")
    if kind == "md":
        return s["plan"].execute_batch(s["y"], s["x"], 1)
    if kind == "md_real":
        s["plan"].execute(s["y"], s["x"], s["temp"])
        s["plan"].execute(s["z"], s["y"], s["temp"])
        return s["y"], s["z"]
    s["plan"].reset()  # a new stream
    for k in range(case["calls"]):
        s["plan"].apply(s["y"][k], s["x"][k])
    return s["y"]


def work(case):
    kind = case["kind"]
    es = {"f32": 4, "f64": 8, "bf16": 2, "f16": 2}[case["dtype"]]

    def fft(n):
        return 5.0 * n * math.log2(max(2, n))

    if kind in ("c2c", "half"):
        passes = 2 if case.get("direction") == "both" else 1
        # the round trip reads the input and writes the spectrum and the result
        tensors = passes + 1
        return {"bytes": tensors * 2 * es * case["n"] * case["batch"], "flops": passes * fft(case["n"]) * case["batch"]}
    if kind == "real":
        n, b = case["n"], case["batch"]
        return {"bytes": b * es * (2 * n + 2 * (n // 2 + 1)), "flops": b * fft(n)}
    if kind == "dct":
        n, b = case["n"], case["batch"]
        return {"bytes": 3 * b * es * n, "flops": b * fft(n)}
    if kind == "conv":
        n, t, b = case["n"], case["taps"], case["batch"]
        h = t * (1 if case["shared"] else b)
        block = 1 << max(8, math.ceil(math.log2(3 * t)))
        # in: signal, taps, output gradient; out: the output and both gradients. Block transforms of the
        # signal and of the gradient, and of the three products (real transforms)
        return {"bytes": es * (b * (2 * n + 2 * (n + t - 1)) + 2 * h),
                "flops": b * n / (block - t + 1) * 5 * fft(block) / 2}
    if kind == "uneven":
        sizes = _lengths(case)[0]
        return {"bytes": 4 * es * int(sizes.sum()), "flops": float(sum(fft(int(n)) for n in sizes))}
    if kind in ("md", "md_real"):
        shape = _shape(case)
        points = math.prod(shape)
        if kind == "md":
            return {"bytes": 4 * es * points, "flops": fft(points)}
        return {"bytes": es * (2 * points + 2 * points // shape[-1] * (shape[-1] // 2 + 1)), "flops": fft(points)}
    t, n = case["taps"], case["block"] * case["calls"]
    block = 1 << math.ceil(math.log2(2 * max(case["block"], t)))
    return {"bytes": es * (2 * n + t), "flops": fft(block) * case["calls"]}


def _dct(x):
    """Unscaled DCT-II and, of its result, DCT-III with the first value halved (rows)."""
    n = x.shape[-1]
    k = torch.arange(n, dtype=torch.float64, device=x.device)
    w = torch.polar(torch.ones_like(k), -math.pi * k / (2 * n))
    y = (torch.fft.fft(torch.cat([x, x.flip(-1)], -1))[..., :n] * w).real / 2
    v = y * w.conj()
    v[..., 0] *= 0.5
    return y, torch.fft.ifft(v, n=2 * n).real[..., :n] * (2 * n)


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "c2c":
        # numpy's transforms take any length without a plan of their own; the GPU takes the large totals
        n = case["n"]
        if n * case["batch"] > 1 << 24:
            x = s["x"].to(torch.complex128)
            f, i = torch.fft.fft, torch.fft.ifft
        else:
            x = s["x"].cpu().numpy().astype(np.complex128)
            f, i = np.fft.fft, np.fft.ifft
        if case["direction"] == "both":
            y = f(x)
            return y, x * n
        return i(x) * n if case["direction"] == "inverse" else f(x)
    if kind == "real":
        x = s["x"].double()
        y = torch.fft.rfft(x) if x.numel() > 1 << 24 else torch.from_numpy(np.fft.rfft(x.cpu().numpy()))
        return y, x * case["n"]
    if kind == "dct":
        x = s["x"].double()
        return _dct(x if x.numel() > 1 << 24 else x.cpu())
    if kind == "conv":
        x, h, g = (s[k].double() for k in "xhg")
        ny = g.shape[-1]
        m = 1 << (ny + case["taps"] - 1).bit_length()
        H, G = torch.fft.rfft(h, m), torch.fft.rfft(g, m)
        X = torch.fft.rfft(x, m)
        y = torch.fft.irfft(X * H, m)[..., :ny]
        dx = torch.fft.irfft(G * H.conj(), m)[..., : case["n"]]
        dh = torch.fft.irfft(G * X.conj(), m)[..., : case["taps"]]
        return y, dx, dh.sum(0) if case["shared"] else dh
    if kind == "uneven":
        x = s["x"].cpu().numpy().astype(np.complex128)
        sizes, inverse = _lengths(case)
        start = np.concatenate([[0], np.cumsum(sizes)[:-1]])
        out = np.empty_like(x)
        for n in np.unique(sizes):
            for d in (0, 1):
                which = start[(sizes == n) & (inverse == d)]
                at = which[:, None] + np.arange(n)
                out[at] = np.fft.ifft(x[at]) * n if d else np.fft.fft(x[at])
        return out
    if kind == "half":
        x = torch.view_as_complex(s["x"].double())
        y = torch.fft.ifft(x) * case["n"] if case["direction"] == "inverse" else torch.fft.fft(x)
        return torch.view_as_real(y)
    if kind == "md":
        return np.fft.fftn(s["x"].cpu().numpy().astype(np.complex128))
    if kind == "md_real":
        x = s["x"].cpu().numpy().astype(np.float64)
        return np.fft.rfftn(x), x * float(x.size)
    x, h = s["x"].double().reshape(-1), s["h"].double()
    m = 1 << (x.numel() + h.numel()).bit_length()
    y = torch.fft.irfft(torch.fft.rfft(x, m) * torch.fft.rfft(h, m), m)[: x.numel()]
    return y.reshape(s["x"].shape)
