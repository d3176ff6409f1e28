"""Performance cases of the 2-D real-to-complex FFT: what users of the package
run, as plain dicts, with the code that prepares, runs and checks one.

A case has a ``kind`` (the public entry point it goes through), a precision and
sizes:

* ``torch``    ``rfft2(x)``: one call of the torch entry point.
* ``plan``     ``Plan(...).exec(in, out)``: a program that keeps its plan and
               buffers (the padded input layout, out of place).
* ``inverse``  ``c2r_2d(X, ny)``: the unnormalised inverse.
* ``train``    ``rfft2_autograd`` and its gradient: one training step's
               transform, forward and backward.
* ``scaled``   ``rfft2_scaled``: FP16 / BF16 storage with power-of-two scales.
* ``batched``  ``BatchedPlan.exec``: uneven FP32 grids, in place.
* ``host``     ``Loop``: the drop-in class on a host buffer, initialize and
               transform, copies included.

All run at the default planning effort ("estimate") unless the case has an
``effort`` of its own.
"""
import math
import os
import random
import sys

import numpy as np
import torch

# the package lies in a folder whose name is not an identifier, under the working folder
_PKG = os.path.join(os.getcwd(), "hpx-fft_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import hpxfft_amd as hp  # noqa: E402
from hpxfft_amd import torch_api  # noqa: E402

_REAL = {"f64": torch.float64, "f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_CPLX = {"f64": torch.complex128, "f32": torch.complex64}
_BYTES = {"f64": 8, "f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # the reference harness's default grid: a call whose cost is launches and host work
        {"name": "small_8x14_f64", "kind": "torch", "prec": "f64", "nx": 8, "ny": 14, "batch": 1},
        # spectral layers on a mini-batch of small images
        {"name": "train_64x128x128_f32", "kind": "train", "prec": "f32", "nx": 128, "ny": 128, "batch": 64},
        # the reference README's grid: few long rows, short columns
        {"name": "plan_256x16384_f64", "kind": "plan", "prec": "f64", "nx": 256, "ny": 16384, "batch": 1},
        # the drop-in class on a host vector, the upper end of the reference's size sweep
        {"name": "host_2048x2048_f64", "kind": "host", "prec": "f64", "nx": 2048, "ny": 2048, "batch": 1},
        # a grid whose sides are not powers of two, small prime factors
        {"name": "plan_3000x3000_f64", "kind": "plan", "prec": "f64", "nx": 3000, "ny": 3000, "batch": 1},
        # sides with a large prime factor, as sizes given by data are (Bluestein on both)
        {"name": "plan_2039x4078_f64", "kind": "plan", "prec": "f64", "nx": 2039, "ny": 4078, "batch": 1},
        # the way back from a spectrum (filtering, solvers), the largest grid of the size sweep
        {"name": "inverse_4096x4096_f64", "kind": "inverse", "prec": "f64", "nx": 4096, "ny": 4096, "batch": 1},
        # sides longer than one workgroup holds that are not powers of two
        {"name": "plan_9000x18000_f64", "kind": "plan", "prec": "f64", "nx": 9000, "ny": 18000, "batch": 1},
        # the headline grid, planned as the benchmark plans it
        {"name": "plan_16384x16384_f64", "kind": "plan", "prec": "f64", "nx": 16384, "ny": 16384, "batch": 1,
         "effort": "measure"},
        # a mini-batch of large images, forward and gradient
        {"name": "train_16x4096x4096_f32", "kind": "train", "prec": "f32", "nx": 4096, "ny": 4096, "batch": 16},
        # a grid kept in half precision, the largest square the plans take
        {"name": "scaled_32768x32768_f16", "kind": "scaled", "prec": "f16", "nx": 32768, "ny": 32768, "batch": 1},
        # many independent grids of uneven sizes in two launches
        {"name": "batched_512_f32", "kind": "batched", "prec": "f32", "count": 512, "shapes": 4},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _length(rng, lo, hi):
    """A side: a power of two, a product of small primes, or (up to 4096) any number."""
    v = _log_uniform(rng, lo, hi)
    style = rng.random()
    if style < 0.35:
        return 1 << max(1, round(math.log2(v)))
    n = max(lo, min(hi, round(v)))
    if style < 0.7 or n > 4096:
        while True:
            m = n
            for f in (2, 3, 5, 7):
                while m % f == 0:
                    m //= f
            if m == 1:
                return n
            n -= 1
    return n


def _sides(rng, lo, hi, points):
    """Nx and Ny/2 of a grid of at most ``points`` points."""
    while True:
        nx, half = _length(rng, lo, hi), _length(rng, lo // 2, hi // 2)
        if nx * 2 * half <= points:
            return nx, half


def draw(rng):
    """One more case of the same ranges: sides of 8 to 16384 (16-bit storage to
    32768, host grids to 2048), batches while a grid is small."""
    kind = rng.choice(["torch", "plan", "plan", "inverse", "train", "scaled", "batched", "host"])
    if kind == "batched":
        return {"kind": kind, "prec": "f32", "count": round(_log_uniform(rng, 8, 512)), "shapes": rng.randrange(1, 1000)}
    if kind == "scaled":
        nx, half = _sides(rng, 16, 32768, 1 << 28)
        return {"kind": kind, "prec": rng.choice(["f16", "bf16"]), "nx": nx, "ny": 2 * half, "batch": 1}
    if kind == "host":
        nx, half = _sides(rng, 8, 2048, 1 << 22)
        return {"kind": kind, "prec": "f64", "nx": nx, "ny": 2 * half, "batch": 1}
    limit = 1 << (26 if kind == "train" else 27)
    nx, half = _sides(rng, 8, 16384, limit)
    most = limit // (nx * 2 * half)
    batch = 1 if kind == "plan" or most < 2 else round(_log_uniform(rng, 1, min(most, 256)))
    return {"kind": kind, "prec": rng.choice(["f64", "f32"]), "nx": nx, "ny": 2 * half, "batch": batch}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _randn(shape, dtype, gen):
    return torch.randn(shape, dtype=dtype, device="cuda", generator=gen)


def _uniform(shape, dtype, gen):
    return torch.empty(shape, dtype=dtype, device="cuda").uniform_(-1.0, 1.0, generator=gen)


def _grids(case):
    """Sides of a batched case's grids (powers of two, 64 to 2048) and their places in one buffer."""
    r = random.Random(case["shapes"])
    sides = [(1 << r.randint(6, 11), 1 << r.randint(6, 11)) for _ in range(case["count"])]
    at, total = [], 0
    for nx, ny in sides:
        at.append(total)
        total += -(-nx * 2 * (ny // 2 + 1) // 64) * 64
    return sides, at, total


def _real_input(case, gen, dtype=None):
    """The real grids (batch, nx, ny) of a torch or train case; images and fields are normal."""
    shape = (case["nx"], case["ny"]) if case["batch"] == 1 else (case["batch"], case["nx"], case["ny"])
    return _randn(shape, dtype or _REAL[case["prec"]], gen)


def _padded_input(case, gen):
    """The padded (nx, 2 (ny/2 + 1)) grid of a plan case, uniform in [-1, 1) as the benchmark's."""
    x = torch.zeros((case["nx"], 2 * (case["ny"] // 2 + 1)), dtype=_REAL[case["prec"]], device="cuda")
    x[:, :case["ny"]] = _uniform((case["nx"], case["ny"]), x.dtype, gen)
    return x


def _spectrum_input(case, gen):
    shape = (case["nx"], case["ny"] // 2 + 1)
    return _randn(shape if case["batch"] == 1 else (case["batch"], *shape), _CPLX[case["prec"]], gen)


def _scaled_input(case, gen):
    """A padded 16-bit grid of normal values."""
    x = torch.zeros((case["nx"], 2 * (case["ny"] // 2 + 1)), dtype=_REAL[case["prec"]], device="cuda")
    x[:, :case["ny"]] = _randn((case["nx"], case["ny"]), x.dtype, gen)
    return x


def _host_input(case, seed):
    x = np.zeros((case["nx"], 2 * (case["ny"] // 2 + 1)))
    x[:, :case["ny"]] = np.random.default_rng(seed).random((case["nx"], case["ny"]))
    return x


def _batched_input(case, gen):
    sides, at, total = _grids(case)
    flat = torch.zeros(total, dtype=torch.float32, device="cuda")
    for (nx, ny), o in zip(sides, at):
        flat[o:o + nx * (ny + 2)].view(nx, ny + 2)[:, :ny].uniform_(-1.0, 1.0, generator=gen)
    return flat


def prepare(case, seed):
    kind = case["kind"]
    if kind == "host":
        return {"case": case, "loop": hp.Loop(), "x": _host_input(case, seed)}
    gen = _gen(seed)
    if kind == "torch":
        return {"case": case, "x": _real_input(case, gen)}
    if kind == "train":
        x = _real_input(case, gen)
        return {"case": case, "x": x.requires_grad_(True), "g": _spectrum_input(case, gen)}
    if kind == "inverse":
        return {"case": case, "X": _spectrum_input(case, gen)}
    if kind == "scaled":
        return {"case": case, "x": _scaled_input(case, gen)}
    if kind == "plan":
        x = _padded_input(case, gen)
        out = torch.empty((case["nx"], case["ny"] // 2 + 1), dtype=_CPLX[case["prec"]], device="cuda")
        plan = hp.Plan(case["nx"], case["ny"], precision=case["prec"], effort=case.get("effort", "estimate"),
                       stream=torch.cuda.current_stream())
        return {"case": case, "x": x, "out": out, "plan": plan}
    sides, at, _ = _grids(case)
    flat = _batched_input(case, gen)
    plan = hp.BatchedPlan([s[0] for s in sides], [s[1] for s in sides], stream=torch.cuda.current_stream())
    return {"case": case, "flat": flat, "plan": plan, "ptrs": [flat.data_ptr() + 4 * o for o in at]}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "torch":
        return torch_api.rfft2(state["x"])
    if kind == "plan":
        state["plan"].exec(state["x"].data_ptr(), state["out"].data_ptr())
        return state["out"]
    if kind == "inverse":
        return torch_api.c2r_2d(state["X"], case["ny"])
    if kind == "train":
        y = torch_api.rfft2_autograd(state["x"])
        (gx,) = torch.autograd.grad(y, state["x"], state["g"])
        return y.detach(), gx
    if kind == "scaled":
        return torch_api.rfft2_scaled(state["x"])
    if kind == "batched":
        state["plan"].exec(state["ptrs"])
        return state["flat"]
    # the reference's program: fill the vector, initialize, transform in place
    loop = state["loop"]
    loop.initialize(state["x"].copy(), "estimate")
    return loop.fft_2d_r2c_par()


def _rfft2_64(x):
    """2-D r2c in FP64, one dimension at a time."""
    return torch.fft.fft(torch.fft.rfft(x.double(), dim=-1), dim=-2)


def exact(case, seed):
    kind = case["kind"]
    if kind == "scaled":
        return None  # stored values carry exponents that the call chooses
    if kind == "host":
        return np.fft.rfft2(_host_input(case, seed)[:, :case["ny"]]).view(np.float64)
    gen = _gen(seed)
    if kind == "torch":
        return _rfft2_64(_real_input(case, gen))
    if kind == "plan":
        return _rfft2_64(_padded_input(case, gen)[:, :case["ny"]].contiguous())
    ny = case.get("ny")
    if kind == "inverse":
        z = torch.fft.ifft(_spectrum_input(case, gen).to(torch.complex128), dim=-2, norm="forward")
        z[..., 0].imag.zero_()
        z[..., -1].imag.zero_()
        return torch.fft.irfft(z, n=ny, dim=-1, norm="forward")
    if kind == "train":
        x = _real_input(case, gen)
        g = _spectrum_input(case, gen).to(torch.complex128)
        # the gradient: Re of the unnormalised inverse transform of g, zero beyond ny/2
        z = torch.fft.ifft(g, dim=-2, norm="forward")
        z[..., 1:-1] *= 0.5
        z[..., 0].imag.zero_()
        z[..., -1].imag.zero_()
        return _rfft2_64(x), torch.fft.irfft(z, n=ny, dim=-1, norm="forward")
    sides, at, total = _grids(case)
    flat = _batched_input(case, gen)
    out = torch.zeros(total, dtype=torch.float64, device="cuda")
    for (nx, ny), o in zip(sides, at):
        n = nx * (ny + 2)
        out[o:o + n] = torch.view_as_real(_rfft2_64(flat[o:o + n].view(nx, ny + 2)[:, :ny].contiguous())).reshape(-1)
    return out


def work(case):
    """Bytes: each input read once, each output written once.  Operations: 2.5 N log2 N of a real N-point grid."""
    def grid(nx, ny, s):
        return nx * ny * s + nx * (ny // 2 + 1) * 2 * s, 2.5 * nx * ny * math.log2(nx * ny)

    if case["kind"] == "batched":
        each = [grid(nx, ny, 4) for nx, ny in _grids(case)[0]]
        return {"bytes": sum(e[0] for e in each), "flops": sum(e[1] for e in each)}
    b, f = grid(case["nx"], case["ny"], _BYTES[case["prec"]])
    times = case["batch"] * (2 if case["kind"] == "train" else 1)
    return {"bytes": b * times, "flops": f * times}
