"""Transforms that a user of this library runs, for timing and for comparing outputs.

Each case is one call (or one operator call) through the public entry points of sip_amd on
data that is already on the GPU, with the plan and the output buffer that a program keeps:

  op       one torch operator call (asd_fft_c2c / asd_fft_r2c / asd_fft_c2r), plan from its cache
  plan     Plan.execute: 1D, 2D and 3D, c2c / r2c / c2r, forward and inverse, any length
  istft    Istft.execute: batched inverse short-time transforms with overlap-add
  ragged   RaggedPlan.execute: one call over transforms of many lengths and two types

listed() holds one or two of every kind of work; draw() picks further sizes of the same ranges:
lengths are powers of two or other products of 2, 3, 5 and 7 (primes in a range of their own),
spread over their logarithm, and the batch follows from a number of points per call.
"""
import math
import random

import numpy as np
import torch

import sip_amd

DEVICE = "cuda"

# points per call (complex points, or real samples) never exceed the largest listed case
MAX_POINTS = 1 << 24


# ------------------------------------------------------------------ cases
def listed():
    return [
        # the operator on a handful of short rows: latency and host time of one call
        {"name": "op_c2c_210x8", "op": "op", "kind": "c2c", "n0": 210, "n1": 0, "n2": 0, "batch": 8, "inverse": False},
        # one ordinary batch of mixed-radix rows (a few MB: launch- and latency-bound)
        {"name": "c2c_1000x256", "op": "plan", "kind": "c2c", "n0": 1000, "n1": 0, "n2": 0, "batch": 256,
         "inverse": False},
        # the plain power-of-two batch
        {"name": "c2c_4096x512", "op": "plan", "kind": "c2c", "n0": 4096, "n1": 0, "n2": 0, "batch": 512,
         "inverse": False},
        # a length with a large prime factor: measured record lengths are not chosen for the FFT
        {"name": "c2c_997x256", "op": "plan", "kind": "c2c", "n0": 997, "n1": 0, "n2": 0, "batch": 256,
         "inverse": False},
        # long lines, back from the spectrum (pulse compression of long records)
        {"name": "c2c_65536x64_inv", "op": "plan", "kind": "c2c", "n0": 65536, "n1": 0, "n2": 0, "batch": 64,
         "inverse": True},
        # spectra of real channels, and the way back at a length that is not a power of two
        {"name": "r2c_8192x1024", "op": "plan", "kind": "r2c", "n0": 8192, "n1": 0, "n2": 0, "batch": 1024,
         "inverse": False},
        {"name": "c2r_2520x1024_inv", "op": "plan", "kind": "c2r", "n0": 2520, "n1": 0, "n2": 0, "batch": 1024,
         "inverse": True},
        # large complex images (2D focusing), and real camera frames of a mixed-radix size
        {"name": "c2c_2048x2048x4", "op": "plan", "kind": "c2c", "n0": 2048, "n1": 2048, "n2": 0, "batch": 4,
         "inverse": False},
        {"name": "r2c_1080x1920x4", "op": "plan", "kind": "r2c", "n0": 1080, "n1": 1920, "n2": 0, "batch": 4,
         "inverse": False},
        # one large volume
        {"name": "c2c_256x256x256", "op": "plan", "kind": "c2c", "n0": 256, "n1": 256, "n2": 256, "batch": 1,
         "inverse": False},
        # resynthesis of 16 channels from their spectrograms
        {"name": "istft_16x1024x1000", "op": "istft", "channel": 16, "nfft": 1024, "frames": 1000, "hop": 256},
        # one batch of 4000 transforms of uneven lengths
        {"name": "ragged_4000_16384", "op": "ragged", "count": 4000, "nmax": 16384, "mix": 1},
    ]


def _smooth(lo, hi):
    """Products of 2, 3, 5 and 7 in [lo, hi], ascending."""
    out = []
    a = 1
    while a <= hi:
        b = a
        while b <= hi:
            c = b
            while c <= hi:
                d = c
                while d <= hi:
                    if d >= lo:
                        out.append(d)
                    d *= 7
                c *= 5
            b *= 3
        a *= 2
    return sorted(out)


def _primes(lo, hi):
    return [p for p in range(max(2, lo), hi + 1) if all(p % q for q in range(2, int(p ** 0.5) + 1))]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _nearest(values, x):
    return min(values, key=lambda v: abs(math.log(v / x)))


def _length(rng, lo, hi, even=False):
    """A length of [lo, hi]: a power of two in two draws of five, else any product of 2, 3, 5, 7."""
    values = [v for v in _smooth(lo, hi) if not (even and v % 2)]
    if rng.random() < 0.4:
        values = [v for v in values if v & (v - 1) == 0]
    return _nearest(values, _log_uniform(rng, lo, hi))


def _batch(rng, points_per_transform, lo, hi):
    return max(1, int(_log_uniform(rng, lo, hi) / points_per_transform))


def draw(rng):
    what = rng.choice(["op", "rows", "rows", "prime", "long", "real", "real", "image", "image", "frames", "volume",
                       "istft", "ragged"])
    inverse = rng.random() < 0.5
    if what == "op":
        kind = rng.choice(["c2c", "r2c", "c2r"])
        n = _length(rng, 16, 4096, even=(kind == "c2r"))
        return {"op": "op", "kind": kind, "n0": n, "n1": 0, "n2": 0, "batch": rng.randint(1, 32),
                "inverse": {"c2c": inverse, "r2c": False, "c2r": True}[kind]}
    if what in ("rows", "prime", "long"):
        if what == "rows":
            n = _length(rng, 32, 16384)
            b = _batch(rng, n, 1 << 14, 1 << 23)
        elif what == "prime":
            n = _nearest(_primes(23, 2039), _log_uniform(rng, 23, 2039))
            b = _batch(rng, n, 1 << 13, (1 << 18) * min(1.0, 997.0 / n))
        else:
            n = _length(rng, 16385, 1 << 20)
            b = _batch(rng, n, 1 << 18, 1 << 23)
        return {"op": "plan", "kind": "c2c", "n0": n, "n1": 0, "n2": 0, "batch": b, "inverse": inverse}
    if what == "real":
        n = _length(rng, 32, 131072)
        return {"op": "plan", "kind": "c2r" if inverse else "r2c", "n0": n, "n1": 0, "n2": 0,
                "batch": _batch(rng, n, 1 << 15, 1 << 23), "inverse": inverse}
    if what == "image":
        x, y = _length(rng, 32, 2048), _length(rng, 32, 2048)
        return {"op": "plan", "kind": "c2c", "n0": x, "n1": y, "n2": 0,
                "batch": _batch(rng, x * y, 1 << 16, MAX_POINTS), "inverse": inverse}
    if what == "frames":
        x, y = _length(rng, 32, 2048), _length(rng, 32, 2048, even=True)
        return {"op": "plan", "kind": "c2r" if inverse else "r2c", "n0": x, "n1": y, "n2": 0,
                "batch": _batch(rng, x * y, 1 << 17, MAX_POINTS), "inverse": inverse}
    if what == "volume":
        while True:
            x, y, z = (_length(rng, 16, 256) for _ in range(3))
            if x * y * z <= MAX_POINTS:
                break
        return {"op": "plan", "kind": "c2c", "n0": x, "n1": y, "n2": z,
                "batch": _batch(rng, x * y * z, 1 << 15, MAX_POINTS), "inverse": inverse}
    if what == "istft":
        nfft = _length(rng, 128, 1280, even=True)
        channel = rng.randint(1, 16)
        frames = int(_log_uniform(rng, 50, 1000))
        return {"op": "istft", "channel": channel, "nfft": nfft, "frames": frames, "hop": nfft // rng.choice([2, 4])}
    return {"op": "ragged", "count": int(_log_uniform(rng, 200, 4000)), "nmax": rng.choice([1024, 2048, 4096, 8192, 16384]),
            "mix": rng.randint(2, 1 << 20)}


# ------------------------------------------------------------------ inputs
def _dims(case):
    return tuple(case[k] for k in ("n0", "n1", "n2") if case[k])


def _rng(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _uniform(shape, g):
    """Complex values, both parts uniform in [-1, 1)."""
    x = torch.rand(tuple(shape) + (2,), generator=g, device=DEVICE, dtype=torch.float32)
    return torch.view_as_complex(x.mul_(2.0).sub_(1.0))


def _signal(shape, g):
    """Real rows: unit Gaussian noise plus one tone of a frequency, amplitude and phase per row."""
    x = torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32)
    n = shape[-1]
    r = torch.rand(tuple(shape[:-1]) + (3,), generator=g, device=DEVICE, dtype=torch.float32)
    f, amp, phase = (r[..., i:i + 1] for i in range(3))
    t = torch.arange(n, device=DEVICE, dtype=torch.float32)
    return x.add_((0.5 + 3.5 * amp) * torch.cos(math.pi * f * t + 2.0 * math.pi * phase))


def _spectrum(dims, batch, g):
    """Half spectra along the last axis; the bins that a real signal has real are real."""
    n = dims[-1]
    x = _uniform((batch,) + dims[:-1] + (n // 2 + 1,), g)
    if len(dims) == 1:
        x.imag[..., 0] = 0.0
        if n % 2 == 0:
            x.imag[..., -1] = 0.0
    return x


def _input(case, g):
    dims, b = _dims(case), case["batch"]
    if case["kind"] == "c2c":
        return _uniform((b,) + dims, g)
    if case["kind"] == "r2c":
        return _signal((b,) + dims, g)
    return _spectrum(dims, b, g)


def _ragged_entries(case):
    """(kind, n, count, inverse) of a ragged batch: lengths log-uniform over the products of 2, 3
    and 5 in [64, nmax], 70% c2c and 30% r2c, forward, transforms of one length together."""
    rng = random.Random(case["mix"])
    lengths = [v for v in _smooth(64, case["nmax"]) if v % 7]
    many = {}
    for _ in range(case["count"]):
        n = _nearest(lengths, _log_uniform(rng, 64, case["nmax"]))
        key = ("c2c" if rng.random() < 0.7 else "r2c", n)
        many[key] = many.get(key, 0) + 1
    return [(kind, n, count, False) for (kind, n), count in sorted(many.items())]


def _ragged_input(extent, g):
    x = torch.rand(extent // 4, generator=g, device=DEVICE, dtype=torch.float32)
    return x.mul_(2.0).sub_(1.0)


def _window(nfft):
    return torch.hann_window(nfft, periodic=True, device=DEVICE, dtype=torch.float32)


# ------------------------------------------------------------------ the calls
def prepare(case, seed):
    g = _rng(seed)
    if case["op"] == "op":
        return {"op": "op", "call": {"c2c": sip_amd.asd_fft_c2c, "r2c": sip_amd.asd_fft_r2c,
                                     "c2r": sip_amd.asd_fft_c2r}[case["kind"]],
                "x": _input(case, g), "forward": not case["inverse"]}
    if case["op"] == "plan":
        plan = sip_amd.Plan(case["kind"], _dims(case), case["batch"], inverse=case["inverse"])
        out = torch.empty(plan.out_shape(), device=DEVICE,
                          dtype=torch.float32 if case["kind"] == "c2r" else torch.complex64)
        return {"op": "plan", "plan": plan, "x": _input(case, g), "out": out}
    if case["op"] == "istft":
        plan = sip_amd.Istft(case["channel"], case["nfft"], case["frames"], case["hop"])
        out = torch.empty((case["channel"], plan.out_len), device=DEVICE, dtype=torch.complex64)
        return {"op": "istft", "plan": plan, "x": _uniform((case["channel"], case["nfft"], case["frames"]), g),
                "window": _window(case["nfft"]), "out": out}
    plan = sip_amd.RaggedPlan(_ragged_entries(case))
    # entries start on 8-byte boundaries: the floats between two of them stay as they are
    return {"op": "ragged", "plan": plan, "x": _ragged_input((plan.in_extent + 7) // 8 * 8, g),
            "out": torch.zeros(plan.out_extent // 4, device=DEVICE, dtype=torch.float32)}


def run(state):
    if state["op"] == "op":
        return state["call"](state["x"], state["forward"])
    if state["op"] == "istft":
        return state["plan"].execute(state["x"], state["window"], out=state["out"])
    if state["op"] == "ragged":
        return state["plan"].execute(state["x"], state["out"])
    return state["plan"].execute(state["x"], out=state["out"])


# ------------------------------------------------------------------ what a pass cannot do without
def _transform_flops(kind, dims, batch):
    points = float(np.prod(dims)) * batch
    return (5.0 if kind == "c2c" else 2.5) * points * math.log2(float(np.prod(dims)))


def _transform_bytes(kind, dims, batch):
    lead = float(np.prod(dims[:-1], dtype=np.float64)) * batch
    n = dims[-1]
    half = n // 2 + 1
    return lead * {"c2c": 16.0 * n, "r2c": 4.0 * n + 8.0 * half, "c2r": 4.0 * n + 8.0 * half}[kind]


def work(case):
    if case["op"] in ("op", "plan"):
        args = case["kind"], _dims(case), case["batch"]
        return {"bytes": _transform_bytes(*args), "flops": _transform_flops(*args)}
    if case["op"] == "istft":
        nfft, frames, hop = case["nfft"], case["frames"], case["hop"]
        out_len = nfft + hop * (frames - 1) - 2 * (nfft // 2)
        points = float(case["channel"]) * nfft * frames
        return {"bytes": 8.0 * points + 8.0 * case["channel"] * out_len + 4.0 * nfft,
                "flops": 5.0 * points * math.log2(nfft) + 4.0 * points}
    rows = _ragged_entries(case)
    return {"bytes": sum(_transform_bytes(kind, (n,), count) for kind, n, count, _ in rows),
            "flops": sum(_transform_flops(kind, (n,), count) for kind, n, count, _ in rows)}


# ------------------------------------------------------------------ the same in 64 bits
def _exact_transform(kind, x, dims, inverse):
    lead = tuple(range(-len(dims), -1))
    if kind == "r2c":
        y = torch.fft.rfft(x.double(), dim=-1)
        return torch.fft.fftn(y, dim=lead) if lead else y
    x = x.to(torch.complex128)
    if kind == "c2c":
        axes = lead + (-1,)
        return torch.fft.ifftn(x, dim=axes, norm="forward") if inverse else torch.fft.fftn(x, dim=axes)
    if lead:
        x = torch.fft.ifftn(x, dim=lead, norm="forward")
    n = dims[-1]
    x.imag[..., 0] = 0.0  # a real signal's first bin, and the last of an even length, are real
    if n % 2 == 0:
        x.imag[..., -1] = 0.0
    return torch.fft.irfft(x, n=n, dim=-1, norm="forward")


def exact(case, seed):
    g = _rng(seed)
    if case["op"] in ("op", "plan"):
        return _exact_transform(case["kind"], _input(case, g).cpu(), _dims(case), case["inverse"])
    if case["op"] == "istft":
        channel, nfft, frames, hop = case["channel"], case["nfft"], case["frames"], case["hop"]
        x = _uniform((channel, nfft, frames), g).cpu().to(torch.complex128)
        w = _window(nfft).cpu().double()
        rows = torch.fft.ifft(x, dim=1).permute(0, 2, 1) * w
        total = nfft + hop * (frames - 1)
        y = torch.zeros((channel, total), dtype=torch.complex128)
        env = torch.zeros(total, dtype=torch.float64)
        for t in range(frames):
            y[:, t * hop:t * hop + nfft] += rows[:, t]
            env[t * hop:t * hop + nfft] += w * w
        crop = slice(nfft // 2, total - nfft // 2)
        return y[:, crop] / env[crop]
    entries = _ragged_entries(case)
    need = sum((_row_bytes(kind, n, "in") * count + 7) // 8 * 8 for kind, n, count, _ in entries)
    last = entries[-1]
    extent = need - ((_row_bytes(last[0], last[1], "in") * last[2] + 7) // 8 * 8
                     - _row_bytes(last[0], last[1], "in") * last[2])
    x = _ragged_input((extent + 7) // 8 * 8, g).cpu()
    at, parts = 0, []
    for kind, n, count, _ in entries:
        words = _row_bytes(kind, n, "in") * count // 4
        v = x[at:at + words]
        v = torch.view_as_complex(v.view(count, n, 2)) if kind == "c2c" else v.view(count, n)
        parts.append(torch.view_as_real(_exact_transform(kind, v, (n,), False)).reshape(-1))
        at += (words + 1) // 2 * 2
    return torch.cat(parts)


def _row_bytes(kind, n, side):
    if kind == "c2c":
        return 8 * n
    return 4 * n if side == "in" else 8 * (n // 2 + 1)
