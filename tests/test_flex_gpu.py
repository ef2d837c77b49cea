"""The flexible-chain kernels (lengths without a compiled chain) against the
FP64 oracle: small and largest lengths, every radix, remainders of a block,
layouts that take them and both directions. Tolerances are the suite's."""
import numpy as np
import pytest

import plfft_amd as P
from plfft_amd import rng
from gpu_util import CPLX_NP, TOL, bf16_bits, bf16_to_f32, from_dev, relerr, to_dev

pytestmark = pytest.mark.gpu

# one to four stages, odd and even, each radix of the engine, both block sizes
LENGTHS = [6, 9, 10, 12, 14, 15, 20, 21, 22, 26, 33, 36, 49, 63, 77, 81, 91, 100, 121, 143, 169, 225,
           360, 1000, 1001, 1344, 2187, 3000, 4095, 5120, 6000, 8190, 10000, 16000]


def _to(torch, z, prec):
    if prec in ("f32", "f64"):
        return to_dev(torch, z.astype(CPLX_NP[prec]))
    r = np.ascontiguousarray(z.astype(np.complex64)).view(np.float32)
    return to_dev(torch, r.astype(np.float16) if prec == "f16" else bf16_bits(r).view(np.int16))


def _from(torch, d, prec):
    a = from_dev(torch, d)
    if prec in ("f32", "f64"):
        return a.astype(np.complex128)
    r = a.astype(np.float32) if prec == "f16" else bf16_to_f32(a.view(np.uint16))
    return r.astype(np.float64).view(np.complex128)


def _round(z, prec, torch):
    return _from(torch, _to(torch, z, prec), prec)


@pytest.mark.parametrize("prec", ["f32", "f64", "f16", "bf16"])
@pytest.mark.parametrize("n", LENGTHS)
def test_c2c_vs_oracle(torch_cuda, orc, prec, n):
    torch = torch_cuda
    if prec == "f64" and n > 8000:
        pytest.skip("beyond one FP64 block")
    # a partial last block; strided with gaps; columns with an odd pitch
    hm = max(3, 2000 // n) + 1
    cols = [(21, 23, 1, 21, 1)] if n <= 4095 else []
    for hm, is_, id_, os_, od_ in [(hm, 1, n, 1, n), (3, 2, 2 * n + 3, 3, 3 * n + 1)] + cols:
        isz, osz = (hm - 1) * id_ + (n - 1) * is_ + 1, (hm - 1) * od_ + (n - 1) * os_ + 1
        x = _round(rng.complex_normal(n + hm, isz), prec, torch)
        d = _to(torch, x, prec)
        for direction in (-1, 1):
            plan = P.Plan("c2c", n, direction, prec, hm, is_, id_, os_, od_)
            assert "flex_c2c" in plan.describe()
            y = _to(torch, np.full(osz, 3 + 4j), prec)
            plan.execute(d, y)
            y = _from(torch, y, prec)
            ref = orc.c2c_batched(x, n, direction, hm, is_, id_, os_, od_, osz)
            hit = (np.arange(hm)[:, None] * od_ + np.arange(n) * os_).ravel()
            assert relerr(y[hit], ref[hit]) < TOL[prec], plan.describe()
            rest = np.ones(osz, bool)
            rest[hit] = False
            assert np.all(y[rest] == 3 + 4j)


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("n", [12, 18, 20, 30, 42, 50, 100, 154, 182, 1000, 1500, 4374, 6000, 10000])
def test_real_vs_oracle(torch_cuda, orc, prec, n):
    """R2C and C2R: packed, odd distances (reals not in pairs), strided."""
    torch = torch_cuda
    m = n // 2 + 1
    rt, ct = (np.float32, np.complex64) if prec == "f32" else (np.float64, np.complex128)
    for hm, is_, id_, os_, od_ in [(7, 1, n, 1, m), (5, 1, n + 1, 1, m + 2), (3, 2, 2 * n + 1, 2, 2 * m)]:
        isz, osz = (hm - 1) * id_ + (n - 1) * is_ + 1, (hm - 1) * od_ + (m - 1) * os_ + 1
        x = rng.normal_f64(n + hm, isz).astype(rt)
        plan = P.Plan("r2c", n, -1, prec, hm, is_, id_, os_, od_)
        assert "flex_r2c" in plan.describe()
        y = to_dev(torch, np.zeros(osz, ct))
        plan.execute(to_dev(torch, x), y)
        ref = orc.r2c_batched(x.astype(np.float64), n, hm, is_, id_, os_, od_, osz)
        hit = (np.arange(hm)[:, None] * od_ + np.arange(m) * os_).ravel()
        assert relerr(from_dev(torch, y)[hit], ref[hit]) < TOL[prec], plan.describe()
        back = P.Plan("c2r", n, 1, prec, hm, os_, od_, is_, id_)
        assert "flex_c2r" in back.describe()
        z = to_dev(torch, np.full(isz, 5, rt))
        back.execute(to_dev(torch, ref.astype(ct)), z)
        z = from_dev(torch, z)
        rhit = (np.arange(hm)[:, None] * id_ + np.arange(n) * is_).ravel()
        assert relerr(z[rhit] / n, x[rhit].astype(np.float64)) < TOL[prec], back.describe()
        rest = np.ones(isz, bool)
        rest[rhit] = False
        assert np.all(z[rest] == 5)


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("kind", ["dct2", "dst2", "dct3", "dst3"])
def test_dct_vs_definition(torch_cuda, prec, kind):
    """Against numpy FP64 sums of the FFTW definitions."""
    torch = torch_cuda
    rt = np.float32 if prec == "f32" else np.float64
    for n, hm, s in ((12, 9, 1), (30, 5, 2), (100, 4, 1), (154, 3, 1), (1000, 3, 1), (1500, 3, 2)):
        x = rng.normal_f64(n, hm * s * n).astype(rt)
        plan = P.Plan("r2r", n, -1, prec, hm, s, s * n, 1, n, r2r=kind)
        assert "flex_dct" in plan.describe()
        y = to_dev(torch, np.zeros(hm * n, rt))
        plan.execute(to_dev(torch, x), y)
        u = x.astype(np.float64).reshape(hm, n, s)[:, :, 0]
        j, k = np.arange(n)[None, :], np.arange(n)[:, None]
        # angles pi i / 2n with the integer reduced mod 4n before the sine
        def cos(i):
            return np.cos(np.pi * (i % (4 * n)) / (2 * n))

        def sin(i):
            return np.sin(np.pi * (i % (4 * n)) / (2 * n))
        if kind == "dct2":
            A = 2 * cos((2 * j + 1) * k)
        elif kind == "dst2":
            A = 2 * sin((2 * j + 1) * (k + 1))
        elif kind == "dct3":
            A = 2 * cos(j * (2 * k + 1))
            A[:, 0] = 1
        else:
            A = 2 * sin((j + 1) * (2 * k + 1))
            A[:, n - 1] = (-1.0) ** np.arange(n)
        ref = u @ A.T
        assert relerr(from_dev(torch, y).reshape(hm, n), ref) < TOL[prec], plan.describe()
