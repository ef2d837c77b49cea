"""The transforms that this library's performance is measured on.

Each case is one thing a user's program does with a plan that it keeps: the
family says which public entry point, the other keys say length, batch, data
type, direction and layout. Inputs are drawn on the GPU from a seed.

Families
  c2c      Plan.execute_async of batched complex transforms ("layout":
           "packed" members back to back, or "columns": member b is column b
           of a row-major n x howmany matrix, both sides)
  sync     the same transform through the drop-in, synchronous Plan.execute
  real     a filter's two halves: R2C of real rows, C2R of a spectrum
  grad     a differentiable transform through torch.autograd: the transform
           of a strided real buffer and the gradient of that buffer
  fixed    Q0.15 / Q0.7 complex transforms
  mixed    MixedPlan.execute_async: a batch whose members differ in length
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "perf-libs-fft_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import plfft_amd as P  # noqa: E402
from plfft_amd import rng as prng  # noqa: E402
from plfft_amd.autograd import PlanFunction  # noqa: E402

_BYTES = {"f32": 4, "f64": 8, "f16": 2, "bf16": 2, "q15": 2, "q7": 1}
_REAL = {"f32": torch.float32, "f64": torch.float64, "f16": torch.float16,
         "bf16": torch.bfloat16}
_CPLX = {"f32": torch.complex64, "f64": torch.complex128}


def listed():
    return [
        # the smallest calls: one frame of a sensor or of audio channels,
        # transformed by an unmodified caller that waits for each result
        {"name": "sync_small", "family": "sync", "n": 1024, "howmany": 16, "dtype": "f32",
         "dir": -1, "layout": "packed"},
        # the benchmark's headline: many medium power-of-two members
        {"name": "c2c_4096", "family": "c2c", "n": 4096, "howmany": 32768, "dtype": "f32",
         "dir": -1, "layout": "packed"},
        # long power-of-two members (spectrum analysis, radar range lines)
        {"name": "c2c_65536", "family": "c2c", "n": 65536, "howmany": 1024, "dtype": "f32",
         "dir": -1, "layout": "packed"},
        # the longest members, double precision, back to the time domain
        # (scientific codes)
        {"name": "c2c_f64_1M", "family": "c2c", "n": 1 << 20, "howmany": 32, "dtype": "f64",
         "dir": 1, "layout": "packed"},
        # a round decimal length, as users choose who do not think in powers
        # of two (sample rates, image sides)
        {"name": "c2c_1000", "family": "c2c", "n": 1000, "howmany": 65536, "dtype": "f32",
         "dir": -1, "layout": "packed"},
        # a long prime length
        {"name": "c2c_65537", "family": "c2c", "n": 65537, "howmany": 512, "dtype": "f32",
         "dir": -1, "layout": "packed"},
        # the second axis of a two-dimensional transform: columns of a matrix
        {"name": "columns_1024", "family": "c2c", "n": 1024, "howmany": 16384, "dtype": "f32",
         "dir": -1, "layout": "columns"},
        # real signals to spectra and spectra back to signals
        {"name": "real_4096", "family": "real", "n": 4096, "howmany": 16384, "dtype": "f32"},
        # a training step's forward and backward through a DCT-II of every
        # second real of a padded buffer
        {"name": "grad_dct2", "family": "grad", "kind": "dct2", "n": 4096, "howmany": 8192,
         "dtype": "f32", "stride": 2, "pad": 64},
        # half-precision storage
        {"name": "c2c_f16_4096", "family": "c2c", "n": 4096, "howmany": 32768, "dtype": "f16",
         "dir": -1, "layout": "packed"},
        # fixed-point storage (embedded signal chains)
        {"name": "q15_4096", "family": "fixed", "n": 4096, "howmany": 32768, "dtype": "q15",
         "dir": -1},
        # members of many lengths, a tenth of them prime
        {"name": "mixed_3000", "family": "mixed", "members": 3000, "lengths_seed": 2024,
         "dtype": "f32", "dir": -1},
    ]


# ---------------------------------------------------------------------------
# more cases of the same ranges
# ---------------------------------------------------------------------------
def _log_int(r, lo, hi):
    return int(round(math.exp(r.uniform(math.log(lo), math.log(hi)))))


def _smooth_near(v):
    """The largest 2^a 3^b 5^c 7^d <= v (a length a user rounds to)."""
    best = 1
    p2 = 1
    while p2 <= v:
        p3 = p2
        while p3 <= v:
            p5 = p3
            while p5 <= v:
                p7 = p5
                while p7 <= v:
                    best = max(best, p7)
                    p7 *= 7
                p5 *= 5
            p3 *= 3
        p2 *= 2
    return best


def _length(r, lo, hi):
    """A length and whether it is a power of two: powers of two, round
    lengths, and lengths that are simply what the data had."""
    v = _log_int(r, lo, hi)
    what = r.random()
    if what < 0.4:
        return 1 << max(lo.bit_length() - 1, min(hi.bit_length() - 1, round(math.log2(v)))), True
    if what < 0.8:
        return max(lo, _smooth_near(v)), False
    return v, False


def draw(rng):
    fam = rng.choice(["c2c", "c2c", "c2c", "c2c", "sync", "real", "real", "grad", "fixed",
                      "mixed"])
    if fam == "c2c":
        dtype = rng.choice(["f32", "f32", "f64", "f16", "bf16"])
        hi = 65536 if dtype in ("f16", "bf16") else 1 << 20
        n, pow2 = _length(rng, 16, hi)
        points = _log_int(rng, 1 << 14, 1 << (26 if pow2 else 24))
        if dtype == "f64":
            points //= 2
        layout = "columns" if n <= 4096 and rng.random() < 0.2 else "packed"
        return {"family": "c2c", "n": n, "howmany": max(1, points // n), "dtype": dtype,
                "dir": rng.choice([-1, 1]), "layout": layout}
    if fam == "sync":
        n, _ = _length(rng, 16, 4096)
        return {"family": "sync", "n": n, "howmany": _log_int(rng, 1, 64),
                "dtype": rng.choice(["f32", "f64"]), "dir": rng.choice([-1, 1]),
                "layout": "packed"}
    if fam == "real":
        dtype = rng.choice(["f32", "f32", "f64"])
        n, pow2 = _length(rng, 16, 1 << 18)
        points = _log_int(rng, 1 << 14, 1 << (25 if pow2 else 23))
        return {"family": "real", "n": n, "howmany": max(1, points // n), "dtype": dtype}
    if fam == "grad":
        n, _ = _length(rng, 16, 16384)
        points = _log_int(rng, 1 << 14, 1 << 24)
        return {"family": "grad", "kind": rng.choice(["dct2", "dst2", "r2c"]), "n": n,
                "howmany": max(1, points // n), "dtype": rng.choice(["f32", "f64"]),
                "stride": rng.choice([1, 2]), "pad": rng.choice([0, 64])}
    if fam == "fixed":
        n = 1 << rng.randint(4, 15)
        points = _log_int(rng, 1 << 14, 1 << 26)
        return {"family": "fixed", "n": n, "howmany": max(1, points // n),
                "dtype": rng.choice(["q15", "q7"]), "dir": rng.choice([-1, 1])}
    return {"family": "mixed", "members": _log_int(rng, 32, 1000),
            "lengths_seed": rng.randrange(1 << 30), "dtype": rng.choice(["f32", "f64", "f16"]),
            "dir": rng.choice([-1, 1])}


# ---------------------------------------------------------------------------
# inputs and plans
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)
    return g


def _normal(count, dtype, g):
    """count reals of a unit-variance signal in the storage type."""
    if dtype in ("q15", "q7"):
        full = 32767 if dtype == "q15" else 127
        x = torch.empty(count, dtype=torch.float32, device="cuda").normal_(generator=g)
        x = (x * (0.25 * full)).round_().clamp_(-full - 1, full)
        return x.to(torch.int16 if dtype == "q15" else torch.int8)
    if dtype in ("f16", "bf16"):
        x = torch.empty(count, dtype=torch.float32, device="cuda").normal_(generator=g)
        return x.to(_REAL[dtype])
    return torch.empty(count, dtype=_REAL[dtype], device="cuda").normal_(generator=g)


def _complex(count, dtype, g):
    """count complex values: a complex tensor (f32, f64) or (re, im) pairs."""
    x = _normal(2 * count, dtype, g).view(count, 2)
    return torch.view_as_complex(x) if dtype in _CPLX else x


def _lengths(case):
    return prng.mixed_lengths(case["lengths_seed"], case["members"])


def _grad_plan(case):
    n, s = case["n"], case["stride"]
    kind, r2r = ("r2c", 0) if case["kind"] == "r2c" else ("r2r", case["kind"])
    return P.Plan(kind, n, P.PLFFT_FORWARD, case["dtype"], howmany=case["howmany"], istride=s,
                  idist=s * n + case["pad"], r2r=r2r)


def prepare(case, seed):
    g = _gen(seed)
    fam, dt = case["family"], case["dtype"]
    st = {"case": case}
    if fam == "mixed":
        lengths = _lengths(case)
        st["plan"] = P.MixedPlan(lengths, case["dir"], dt)
        st["x"] = _complex(sum(lengths), dt, g)
        st["y"] = torch.empty_like(st["x"])
        st["ws"] = torch.empty(max(1, st["plan"].workspace_size), dtype=torch.uint8,
                               device="cuda")
        return st
    n, hm = case["n"], case["howmany"]
    if fam in ("c2c", "sync", "fixed"):
        lay = {}
        if case.get("layout") == "columns":
            lay = {"istride": hm, "idist": 1, "ostride": hm, "odist": 1}
        st["plan"] = P.Plan("c2c", n, case["dir"], dt, howmany=hm, **lay)
        st["x"] = _complex(n * hm, dt, g)
        st["y"] = torch.empty_like(st["x"])
    elif fam == "real":
        st["r2c"] = P.Plan("r2c", n, P.PLFFT_FORWARD, dt, howmany=hm)
        st["c2r"] = P.Plan("c2r", n, P.PLFFT_BACKWARD, dt, howmany=hm)
        st["x"] = _normal(n * hm, dt, g)
        st["X"] = torch.empty(hm * (n // 2 + 1), dtype=_CPLX[dt], device="cuda")
        # the spectrum that goes back: of a real signal, as a filter leaves it
        st["F"] = _complex(hm * (n // 2 + 1), dt, g)
        F = st["F"].view(hm, n // 2 + 1)
        F[:, 0].imag.zero_()
        if n % 2 == 0:
            F[:, n // 2].imag.zero_()
        st["z"] = torch.empty(n * hm, dtype=_REAL[dt], device="cuda")
    elif fam == "grad":
        st["plan"] = _grad_plan(case)
        st["x"] = _normal(hm * (case["stride"] * n + case["pad"]), dt, g).requires_grad_()
        count = hm * (n // 2 + 1 if case["kind"] == "r2c" else n)
        st["gy"] = _complex(count, dt, g) if case["kind"] == "r2c" else _normal(count, dt, g)
    else:
        raise ValueError(fam)
    return st


def run(state):
    fam = state["case"]["family"]
    if fam == "sync":
        state["plan"].execute(state["x"], state["y"])
        return state["y"]
    stream = torch.cuda.current_stream()
    if fam in ("c2c", "fixed"):
        state["plan"].execute_async(state["x"], state["y"], stream=stream)
        return state["y"]
    if fam == "mixed":
        state["plan"].execute_async(state["x"], state["y"], stream=stream,
                                    workspace=state["ws"])
        return state["y"]
    if fam == "real":
        state["r2c"].execute_async(state["x"], state["X"], stream=stream)
        state["c2r"].execute_async(state["F"], state["z"], stream=stream)
        return state["X"], state["z"]
    y = PlanFunction.apply(state["x"], state["plan"])
    (gx,) = torch.autograd.grad(y, state["x"], state["gy"])
    return y.detach(), gx


# ---------------------------------------------------------------------------
# the work no implementation can do without, and the exact values
# ---------------------------------------------------------------------------
def work(case):
    fam, b = case["family"], _BYTES[case["dtype"]]
    if fam == "mixed":
        lengths = _lengths(case)
        return {"bytes": 4 * b * sum(lengths),
                "flops": sum(5.0 * n * math.log2(n) for n in lengths)}
    n, hm = case["n"], case["howmany"]
    full = 5.0 * n * math.log2(n) * hm
    if fam in ("c2c", "sync", "fixed"):
        return {"bytes": 4 * b * n * hm, "flops": full}
    spec = 2 * b * (n // 2 + 1) * hm
    if fam == "real":
        return {"bytes": 2 * (b * n * hm + spec), "flops": full}
    # grad: the strided input's elements, the output, its gradient, and the
    # whole gradient buffer
    out = spec if case["kind"] == "r2c" else b * n * hm
    return {"bytes": b * n * hm + 2 * out + b * hm * (case["stride"] * n + case["pad"]),
            "flops": full}


def _host64(x):
    """(re, im) pairs or a complex tensor as complex128 on the host."""
    if not x.is_complex():
        x = torch.view_as_complex(x.cpu().to(torch.float64).contiguous())
    return x.cpu().to(torch.complex128)


def _dft64(x, direction):
    """Unnormalized DFT of the rows of x, complex128."""
    return torch.fft.fft(x) if direction < 0 else torch.fft.ifft(x, norm="forward")


def _pairs_if(y, dtype):
    return y if dtype in _CPLX else torch.view_as_real(y)


def exact(case, seed):
    fam, dt = case["family"], case["dtype"]
    if fam == "fixed":
        return None  # whole numbers
    st = prepare(case, seed)
    if fam == "mixed":
        x = _host64(st["x"])
        y = torch.empty_like(x)
        o = 0
        for n in _lengths(case):
            y[o:o + n] = _dft64(x[o:o + n], case["dir"])
            o += n
        return _pairs_if(y, dt)
    n, hm = case["n"], case["howmany"]
    if fam in ("c2c", "sync"):
        x = _host64(st["x"])
        if case["layout"] == "columns":
            y = _dft64(x.view(n, hm).t(), case["dir"]).t().contiguous()
        else:
            y = _dft64(x.view(hm, n), case["dir"])
        return _pairs_if(y.reshape(-1), dt)
    if fam == "real":
        x = st["x"].cpu().to(torch.float64).view(hm, n)
        X = torch.fft.rfft(x).reshape(-1)
        F = _host64(st["F"]).view(hm, n // 2 + 1)
        return X, torch.fft.irfft(F, n=n, norm="forward").reshape(-1)
    # grad
    s, pad = case["stride"], case["pad"]
    x = st["x"].detach().cpu().to(torch.float64).view(hm, s * n + pad)
    u = x[:, :s * n:s].contiguous()
    gx = torch.zeros_like(x)
    if case["kind"] == "r2c":
        y = torch.fft.rfft(u)
        G = _host64(st["gy"]).view(hm, n // 2 + 1)
        full = torch.zeros(hm, n, dtype=torch.complex128)
        full[:, :n // 2 + 1] = G
        gx[:, :s * n:s] = torch.fft.ifft(full, norm="forward").real
        return y.reshape(-1), gx.reshape(-1)
    G = st["gy"].cpu().to(torch.float64).view(hm, n)
    dst = case["kind"] == "dst2"
    sign = torch.ones(n, dtype=torch.float64)
    if dst:  # DST-II(u)_k = DCT-II((-1)^j u)_{n-1-k}
        sign[1::2] = -1.0
        G = G.flip(1)
    w = torch.polar(torch.ones(n, dtype=torch.float64),
                    -math.pi / (2 * n) * torch.arange(n, dtype=torch.float64))
    v = u * sign
    y = (torch.fft.fft(torch.cat([v, v.flip(1)], 1))[:, :n] * w).real
    if dst:
        y = y.flip(1)
    full = torch.zeros(hm, 2 * n, dtype=torch.complex128)
    full[:, :n] = G * w.conj()
    gx[:, :s * n:s] = 2.0 * torch.fft.ifft(full, norm="forward").real[:, :n] * sign
    return y.reshape(-1), gx.reshape(-1)
