"""The calls a program using this FFT engine makes, as cases to be timed.

A case is a dict of plain values.  ``kind`` names the entry point:

* ``c2c``       complex transform over some axes through ``DataDesc`` / ``FFTDesc`` / ``apply``;
* ``real``      r2c of a real array and c2r back, through the same descriptors (what a filter
                in the frequency domain does on either side of its product);
* ``dct``       a cosine (or sine) transform and its inverse through ``DCTDesc`` / ``apply``;
* ``host``      the 1-D ``fft`` / ``ifft`` overloads on host arrays;
* ``ragged``    one packed batch of many real signals of unequal lengths (``RaggedBatch``);
* ``mfma``      complex64 rows on the matrix cores (``MfmaFFT``);
* ``conv``      ``fft_conv2d`` of an image batch with its backward pass;
* ``resample``  ``resample`` of a device signal with a given filter.

Shapes and axes are written as text ("16x1080x1920", "1,2").
"""
import math

import numpy as np
import torch

from impulse_amd import autograd as AG
from impulse_amd import fft as F
from impulse_amd import synth
from impulse_amd.mfma import MfmaFFT
from impulse_amd.ragged import RaggedBatch
from impulse_amd.signal import generate_resampling_filter, resample

_REAL = {"f64": torch.float64, "f32": torch.float32}
_COMPLEX = {"f64": torch.complex128, "f32": torch.complex64}
_INVERSE = {1: 1, 2: 3, 3: 2, 4: 4}


def listed():
    return [
        # the smallest call: one short spectrum, where the launch and the call around it are the time
        {"name": "c2c_1000", "kind": "c2c", "shape": "1x1000", "axes": "1", "dtype": "f64", "forward": True},
        # the Nim fft(seq) overload: host data in, host data out
        {"name": "host_fft_8191", "kind": "host", "n": 8191, "complex": False},
        # a block of odd-length real rows (the reference's own CPU-sized workload)
        {"name": "real_256x4095", "kind": "real", "shape": "256x4095", "axes": "1", "dtype": "f64"},
        # the complex 2-D transform at scale
        {"name": "c2c_4096x4096", "kind": "c2c", "shape": "4096x4096", "axes": "0,1", "dtype": "f64",
         "forward": True},
        # long real signals, longer than one workgroup's LDS holds
        {"name": "real_16x4194304", "kind": "real", "shape": "16x4194304", "axes": "1", "dtype": "f64"},
        # long signals of prime length (Bluestein)
        {"name": "real_4x1000003", "kind": "real", "shape": "4x1000003", "axes": "1", "dtype": "f64"},
        # a batch of float32 HD images, both axes, lengths that are not powers of two
        {"name": "real_16x1080x1920_f32", "kind": "real", "shape": "16x1080x1920", "axes": "1,2", "dtype": "f32"},
        # image coefficients (DCT-II) and back (DCT-III) of one 4K frame
        {"name": "dct_2160x3840", "kind": "dct", "shape": "2160x3840", "axes": "0,1", "type": 2, "sine": False},
        # thousands of signals of unequal lengths in one packed buffer
        {"name": "ragged_4000", "kind": "ragged", "count": 4000, "lo": 64, "hi": 262144, "smooth": 0.7, "lengths": 0},
        # complex64 rows on the matrix cores
        {"name": "mfma_2048x65536", "kind": "mfma", "length": 65536, "batch": 2048, "precision": "f32"},
        # one training step's worth of a large-kernel image convolution: forward and both gradients
        {"name": "conv_16x2048x2048_63x63", "kind": "conv", "batch": 16, "height": 2048, "width": 2048, "kh": 63,
         "kw": 63, "dtype": "f32"},
        # rate conversion 44.1 kHz -> 48 kHz of 95 s of audio
        {"name": "resample_160_147", "kind": "resample", "n": 1 << 22, "up": 160, "down": 147, "factor": 10,
         "dtype": "f64"},
    ]


# ---------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------

def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _smooth(n, primes):
    """The largest number <= n whose prime factors are all in `primes` (n >= 1)."""
    for m in range(n, 0, -1):
        r = m
        for p in primes:
            while r % p == 0:
                r //= p
        if r == 1:
            return m
    return 1


def _length(rng, lo, hi):
    """A transform length in [lo, hi]: a power of two, a smooth number or any number."""
    n = _log_int(rng, lo, hi)
    how = rng.random()
    if how < 0.25:
        return max(lo, 1 << (n.bit_length() - 1))
    if how < 0.75:
        return max(lo, _smooth(n, (2, 3, 5, 7, 11, 13)))
    return n


def _array(rng):
    """Shape and axes of a batch of 1-D, 2-D or 3-D transforms, at most 2^24 points."""
    total = 1 << 24
    rank = rng.choice((1, 1, 2, 2, 3))
    if rank == 1:
        # most 1-D work is many short rows; some is few long ones
        n = _length(rng, 64, 16384) if rng.random() < 0.7 else _length(rng, 16384, 1 << 21)
        lens = [n]
    elif rank == 2:
        lens = [_length(rng, 32, 3072), _length(rng, 32, 4096)]
    else:
        lens = [_length(rng, 16, 256) for _ in range(3)]
    size = math.prod(lens)
    batch = _log_int(rng, 1, max(1, total // size))
    return "x".join(str(v) for v in [batch] + lens), ",".join(str(1 + i) for i in range(rank))


def draw(rng):
    kind = rng.choice(("c2c", "c2c", "real", "real", "real", "dct", "host", "ragged", "mfma", "conv", "resample"))
    if kind == "c2c":
        shape, axes = _array(rng)
        return {"kind": kind, "shape": shape, "axes": axes, "dtype": rng.choice(("f64", "f32")),
                "forward": rng.random() < 0.5}
    if kind == "real":
        shape, axes = _array(rng)
        return {"kind": kind, "shape": shape, "axes": axes, "dtype": rng.choice(("f64", "f32"))}
    if kind == "dct":
        h, w = _length(rng, 16, 2160), _length(rng, 64, 4096)
        batch = _log_int(rng, 1, max(1, (1 << 23) // (h * w)))
        return {"kind": kind, "shape": f"{batch}x{h}x{w}", "axes": rng.choice(("2", "1,2")),
                "type": rng.choice((2, 2, 3, 4)), "sine": rng.random() < 0.25}
    if kind == "host":
        return {"kind": kind, "n": _length(rng, 64, 262144), "complex": rng.random() < 0.5}
    if kind == "ragged":
        lo = _log_int(rng, 32, 1024)
        return {"kind": kind, "count": _log_int(rng, 100, 4000), "lo": lo, "hi": _log_int(rng, 4096, 262144),
                "smooth": rng.choice((0.5, 0.7, 0.9, 1.0)), "lengths": rng.randrange(1 << 20)}
    if kind == "mfma":
        length = 1 << rng.randrange(8, 21)
        return {"kind": kind, "length": length, "batch": _log_int(rng, 1, max(1, (1 << 27) // length)),
                "precision": rng.choice(("f32", "f32", "bf16x"))}
    if kind == "conv":
        h, w = _log_int(rng, 128, 2048), _log_int(rng, 128, 2048)
        return {"kind": kind, "batch": _log_int(rng, 1, max(1, min(32, (1 << 26) // (h * w)))), "height": h,
                "width": w, "kh": rng.randrange(7, 64), "kw": rng.randrange(7, 64),
                "dtype": rng.choice(("f32", "f64"))}
    up, down = rng.choice(((3, 2), (2, 3), (160, 147), (147, 160), (1, 4), (4, 1), (1, 2), (320, 441)))
    return {"kind": "resample", "n": _log_int(rng, 1 << 12, 1 << 22), "up": up, "down": down,
            "factor": rng.choice((5, 10, 20)), "dtype": rng.choice(("f64", "f32"))}


# ---------------------------------------------------------------------------
# inputs, plans and passes
# ---------------------------------------------------------------------------

def _ints(text, sep):
    return [int(v) for v in text.split(sep)]


def _gen(seed, device):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _uniform(shape, dtype, seed):
    """Samples in [-1, 1)."""
    return torch.rand(shape, dtype=dtype, device="cuda", generator=_gen(seed, "cuda")).mul_(2).sub_(1)


def _normal(shape, dtype, seed):
    return torch.randn(shape, dtype=dtype, device="cuda", generator=_gen(seed, "cuda"))


def _half(shape, axis):
    return [v // 2 + 1 if i == axis else v for i, v in enumerate(shape)]


def _points(shape, axes):
    return math.prod(shape[a] for a in axes)


def _dct_logical(n, kind, sine):
    return 2 * ((n + 1 if sine else n - 1) if kind == 1 else n)


def _ragged_lengths(case):
    return synth.ragged_lengths(case["count"], case["lo"], case["hi"], case["smooth"], seed=case["lengths"])


def _filter(case):
    return generate_resampling_filter(case["up"], case["down"], case["factor"])


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "c2c":
        shape = _ints(case["shape"], "x")
        s.update(shape=shape, axes=_ints(case["axes"], ","), forward=case["forward"])
        s["x"] = _normal(shape, _COMPLEX[case["dtype"]], seed)
        s["y"] = torch.empty_like(s["x"])
        s["fct"] = 1.0 if case["forward"] else 1.0 / _points(shape, s["axes"])
    elif kind == "real":
        shape, axes = _ints(case["shape"], "x"), _ints(case["axes"], ",")
        s.update(shape=shape, axes=axes, half=_half(shape, axes[-1]), fct=1.0 / _points(shape, axes))
        s["x"] = _uniform(shape, _REAL[case["dtype"]], seed)
        s["y"] = torch.empty(s["half"], dtype=_COMPLEX[case["dtype"]], device="cuda")
        s["z"] = torch.empty_like(s["x"])
    elif kind == "dct":
        shape, axes = _ints(case["shape"], "x"), _ints(case["axes"], ",")
        s.update(shape=shape, axes=axes, type=case["type"], sine=case["sine"])
        s["fct"] = 1.0 / math.prod(_dct_logical(shape[a], case["type"], case["sine"]) for a in axes)
        s["x"] = _uniform(shape, torch.float64, seed)
        s["y"], s["z"] = torch.empty_like(s["x"]), torch.empty_like(s["x"])
    elif kind == "host":
        rng = np.random.default_rng(int(seed))
        x = rng.uniform(-1.0, 1.0, case["n"])
        s["x"] = x + 1j * rng.uniform(-1.0, 1.0, case["n"]) if case["complex"] else x
    elif kind == "ragged":
        s["plan"] = RaggedBatch(_ragged_lengths(case))
        s["x"] = _uniform([s["plan"].in_elems], torch.float32, seed)
        s["y"] = torch.empty(s["plan"].out_elems, dtype=torch.complex128, device="cuda")
    elif kind == "mfma":
        s["plan"] = MfmaFFT(case["length"], case["batch"], case["precision"])
        s["x"] = _normal([case["batch"], case["length"]], torch.complex64, seed)
        s["y"] = torch.empty(s["x"].shape, dtype=s["plan"].out_dtype, device="cuda")
    elif kind == "conv":
        dt = _REAL[case["dtype"]]
        shape, ks = [case["batch"], case["height"], case["width"]], [case["kh"], case["kw"]]
        s["x"] = torch.rand(shape, dtype=dt, device="cuda", generator=_gen(seed, "cuda")).requires_grad_()
        s["k"] = (_normal(ks, dt, seed + 1000003) / math.sqrt(ks[0] * ks[1])).requires_grad_()
        s["g"] = _normal(shape, dt, seed + 2000003)
    else:
        s["x"] = _uniform([case["n"]], _REAL[case["dtype"]], seed)
        s.update(h=_filter(case), up=case["up"], down=case["down"])
    return s


def run(s):
    kind = s["kind"]
    if kind == "c2c":
        F.apply(F.FFTDesc(s["axes"], s["forward"], s["fct"]), F.DataDesc(s["y"], s["shape"]),
                F.DataDesc(s["x"], s["shape"]))
        return s["y"]
    if kind == "real":
        F.apply(F.FFTDesc(s["axes"], True), F.DataDesc(s["y"], s["half"]), F.DataDesc(s["x"], s["shape"]))
        F.apply(F.FFTDesc(s["axes"], False, s["fct"]), F.DataDesc(s["z"], s["shape"]), F.DataDesc(s["y"], s["half"]))
        return s["y"], s["z"]
    if kind == "dct":
        x, y, z = (F.DataDesc(s[v], s["shape"]) for v in "xyz")
        F.apply(F.DCTDesc(s["axes"], s["type"], sine=s["sine"]), y, x)
        F.apply(F.DCTDesc(s["axes"], _INVERSE[s["type"]], False, s["fct"], sine=s["sine"]), z, y)
        return s["y"], s["z"]
    if kind == "host":
        y = F.fft(s["x"], True)
        return y, F.ifft(y)
    if kind == "ragged":
        return s["plan"].execute(s["x"], s["y"])
    if kind == "mfma":
        return s["plan"](s["x"], s["y"])
    if kind == "conv":
        y = AG.fft_conv2d(s["x"], s["k"])
        gx, gk = torch.autograd.grad(y, (s["x"], s["k"]), s["g"])
        return y.detach(), gx, gk
    return resample(s["x"], s["h"], s["up"], s["down"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _log2(n):
    return math.log2(n) if n > 1 else 0.0


def work(case):
    kind = case["kind"]
    if kind in ("c2c", "real", "dct"):
        shape, axes = _ints(case["shape"], "x"), _ints(case["axes"], ",")
        size = math.prod(shape)
        flops = 5.0 * size * sum(_log2(shape[a]) for a in axes)
        if kind == "c2c":
            return {"bytes": 2 * size * (16 if case["dtype"] == "f64" else 8), "flops": flops}
        b = 8 if kind == "dct" or case["dtype"] == "f64" else 4
        if kind == "dct":
            return {"bytes": 4 * size * b, "flops": flops}
        half = math.prod(_half(shape, axes[-1]))
        return {"bytes": 2 * (size * b + half * 2 * b), "flops": flops}
    if kind == "host":
        n = case["n"]
        return {"bytes": (16 if case["complex"] else 8) * n + 48 * n,
                "flops": (10.0 if case["complex"] else 7.5) * n * _log2(n)}
    if kind == "ragged":
        n = _ragged_lengths(case)
        return {"bytes": float(np.sum(4 * n + 16 * (n // 2 + 1))), "flops": float(np.sum(2.5 * n * np.log2(n)))}
    if kind == "mfma":
        n = case["length"] * case["batch"]
        return {"bytes": n * (8 + (8 if case["precision"] == "f32" else 16)), "flops": 5.0 * n * _log2(case["length"])}
    if kind == "conv":
        b = 4 if case["dtype"] == "f32" else 8
        img, k = case["batch"] * case["height"] * case["width"], case["kh"] * case["kw"]
        grid = (case["height"] + case["kh"] - 1) * (case["width"] + case["kw"] - 1)
        # five real transforms of every image (x and y forward; x, g and gx backward)
        return {"bytes": b * (5 * img + 3 * k), "flops": 12.5 * case["batch"] * grid * _log2(grid)}
    nout = math.ceil(case["n"] * case["up"] / case["down"])
    taps = 2 * case["factor"] * max(case["up"], case["down"]) + 1
    b = 4 if case["dtype"] == "f32" else 8
    return {"bytes": b * (case["n"] + nout) + 8 * taps, "flops": 2.0 * nout * taps / case["up"]}


# ---------------------------------------------------------------------------
# the same values in 64 bits, on the CPU
# ---------------------------------------------------------------------------

def _wide(t):
    t = t.detach().cpu()
    return t.to(torch.complex128 if t.is_complex() else torch.float64)


def _dct_matrix(n, kind, sine):
    """M with out = M @ x for the unnormalised transform of type `kind`."""
    i = torch.arange(n, dtype=torch.int64)
    k, j = i[:, None], i[None, :]
    per = 8 * n if kind == 4 else 4 * n
    if kind == 1:
        per = 2 * (n + 1) if sine else 2 * (n - 1)
        a = (k + 1) * (j + 1) if sine else k * j
    elif kind == 2:
        a = (k + 1) * (2 * j + 1) if sine else k * (2 * j + 1)
    elif kind == 3:
        a = (2 * k + 1) * (j + 1) if sine else (2 * k + 1) * j
    else:
        a = (2 * k + 1) * (2 * j + 1)
    ang = (a % per).to(torch.float64) * (2.0 * math.pi / per)
    m = 2.0 * (torch.sin(ang) if sine else torch.cos(ang))
    # the end points that the even or odd extension meets once
    if not sine and kind in (1, 3):
        m[:, 0] *= 0.5
    if not sine and kind == 1:
        m[:, n - 1] *= 0.5
    if sine and kind == 3:
        m[:, n - 1] *= 0.5
    return m


def _dct_over(x, axes, kind, sine):
    for a in axes:
        x = torch.movedim(torch.movedim(x, a, -1) @ _dct_matrix(x.shape[a], kind, sine).T, -1, a)
    return x.contiguous()


def _conv_exact(x, k, g):
    (B, H, W), (KH, KW) = x.shape, k.shape
    P, Q = _smooth_up(H + KH - 1), _smooth_up(W + KW - 1)
    cy, cx = (KH - 1) // 2, (KW - 1) // 2
    kf = torch.fft.rfft2(k, s=(P, Q))
    y, gx, gk = torch.empty_like(x), torch.empty_like(x), torch.zeros(P, Q // 2 + 1, dtype=torch.complex128)
    for b in range(B):
        xf = torch.fft.rfft2(x[b], s=(P, Q))
        y[b] = torch.fft.irfft2(xf * kf, s=(P, Q))[cy:cy + H, cx:cx + W]
        full = torch.zeros(P, Q, dtype=torch.float64)
        full[cy:cy + H, cx:cx + W] = g[b]
        gf = torch.fft.rfft2(full)
        gx[b] = torch.fft.irfft2(gf * kf.conj(), s=(P, Q))[:H, :W]
        gk += gf * xf.conj()
    return y, gx, torch.fft.irfft2(gk, s=(P, Q))[:KH, :KW].contiguous()


def _smooth_up(n):
    while _smooth(n, (2, 3, 5, 7)) != n:
        n += 1
    return n


def _resample_exact(x, h, up, down):
    """Output j is sample (j + delay) down of the full convolution of the zero-stuffed signal with
    the taps behind `lead` zeros, where lead and delay put the middle tap on a kept sample."""
    n, nh = x.shape[0], len(h)
    mid = (nh - 1) / 2.0
    lead = int(math.floor(down - (mid - down * math.floor(mid / down))))
    delay = int(math.ceil(mid + lead)) // down
    m = (torch.arange(math.ceil(n * up / down), dtype=torch.int64) + delay) * down - lead
    q, r = torch.div(m, up, rounding_mode="floor"), torch.remainder(m, up)
    taps = torch.zeros(-(-nh // up) * up, dtype=torch.float64)
    taps[:nh] = torch.from_numpy(np.asarray(h, np.float64))
    if (taps.numel() // up) * m.numel() > 1 << 30:
        return None
    y = torch.zeros(m.numel(), dtype=torch.float64)
    for l in range(taps.numel() // up):
        at = q - l
        y += torch.where((at >= 0) & (at < n), x[at.clamp(0, n - 1)], 0.0) * taps[r + l * up]
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind == "mfma" and case["length"] * case["batch"] > 1 << 28:
        return None
    s = prepare(case, seed)
    if kind == "c2c":
        x = _wide(s["x"])
        return torch.fft.fftn(x, dim=s["axes"]) if s["forward"] else torch.fft.ifftn(x, dim=s["axes"])
    if kind == "real":
        x = _wide(s["x"])
        return torch.fft.rfftn(x, dim=s["axes"]), x
    if kind == "dct":
        x = _wide(s["x"])
        return _dct_over(x, s["axes"], s["type"], s["sine"]), x
    if kind == "host":
        return np.fft.fft(s["x"]), s["x"].astype(np.complex128)
    if kind == "ragged":
        x = _wide(s["x"])
        return torch.cat([torch.fft.rfft(x[i:i + n]) for i, n in
                          zip(s["plan"].in_offsets.tolist(), s["plan"].lengths.tolist())])
    if kind == "mfma":
        return torch.fft.fft(_wide(s["x"]))
    if kind == "conv":
        return _conv_exact(_wide(s["x"]), _wide(s["k"]), _wide(s["g"]))
    return _resample_exact(_wide(s["x"]), s["h"], s["up"], s["down"])
