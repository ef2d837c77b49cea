"""Layouts and directions of the flexible-chain kernels: in place, the adjoints
of the cosine and sine transforms, columns of many tiles; and short real members
of a batch large enough to pass through LDS.

Tolerances are the suite's: relative L2 of 2e-6 (FP32), 1e-13 (FP64).
"""
import numpy as np
import pytest
import scipy.fft as sf

import plfft_amd as P
from plfft_amd import rng
from gpu_util import CPLX_NP, TOL, from_dev, relerr, to_dev

pytestmark = pytest.mark.gpu
REAL = {"f32": np.float32, "f64": np.float64}
PRECS = pytest.mark.parametrize("prec", ["f32", "f64"])


@PRECS
@pytest.mark.parametrize("n", [6, 60, 100, 1000, 3000])
def test_in_place_c2c(torch_cuda, prec, n):
    hm = 4000 // n + 3
    x = rng.complex_normal(n, hm * (n + 1)).astype(CPLX_NP[prec]).reshape(hm, n + 1)
    for direction, f in ((-1, np.fft.fft), (1, np.fft.ifft)):
        plan = P.Plan("c2c", n, direction, prec, hm, 1, n + 1, 1, n + 1, may_alias=True)
        assert "flex_c2c" in plan.describe()
        d = to_dev(torch_cuda, x)
        plan.execute(d, d)
        y = from_dev(torch_cuda, d)
        ref = f(x[:, :n].astype(complex)) * (n if direction > 0 else 1)
        assert relerr(y[:, :n], ref) < TOL[prec], plan.describe()
        assert np.array_equal(y[:, n], x[:, n])


@PRECS
@pytest.mark.parametrize("n", [12, 100, 1000, 6000])
def test_in_place_real(torch_cuda, prec, n):
    """Rows of n + 2 reals that hold the n / 2 + 1 bins as well."""
    hm, m = 4000 // n + 3, n // 2 + 1
    x = rng.normal_f64(n, hm * 2 * m).astype(REAL[prec]).reshape(hm, 2 * m)
    r2c = P.Plan("r2c", n, -1, prec, hm, 1, 2 * m, 1, m, may_alias=True)
    c2r = P.Plan("c2r", n, 1, prec, hm, 1, m, 1, 2 * m, may_alias=True)
    assert "flex_r2c" in r2c.describe() and "flex_c2r" in c2r.describe()
    d = to_dev(torch_cuda, x)
    r2c.execute(d, d)
    ref = np.fft.rfft(x[:, :n].astype(np.float64))
    assert relerr(from_dev(torch_cuda, d).view(CPLX_NP[prec]), ref) < TOL[prec]
    d = to_dev(torch_cuda, ref.astype(CPLX_NP[prec]).view(REAL[prec]))
    c2r.execute(d, d)
    assert relerr(from_dev(torch_cuda, d)[:, :n] / n, x[:, :n]) < TOL[prec]


@PRECS
@pytest.mark.parametrize("kind,type_,sine", [("dct2", 2, 0), ("dct3", 3, 0), ("dst2", 2, 1), ("dst3", 3, 1)])
@pytest.mark.parametrize("n", [30, 100, 1000])
def test_adjoint_of_r2r(torch_cuda, prec, kind, type_, sine, n):
    """<T x, y> = <x, T^t y>: T^t of the unit vectors' transforms, in FP64."""
    A = (sf.dst if sine else sf.dct)(np.eye(n), type=type_, axis=0)
    for hm in (1, 5, 700):
        y = rng.normal_f64(n + hm, hm * n).astype(REAL[prec])
        plan = P.Plan("r2r", n, -1, prec, hm, r2r=kind)
        assert "flex_dct" in plan.describe()
        x = to_dev(torch_cuda, np.zeros(hm * n, REAL[prec]))
        plan.adjoint(to_dev(torch_cuda, y), x)
        ref = y.astype(np.float64).reshape(hm, n) @ A
        assert relerr(from_dev(torch_cuda, x).reshape(hm, n), ref) < TOL[prec], plan.describe()


@PRECS
@pytest.mark.parametrize("n,cols", [(100, 4099), (60, 1000), (1000, 333), (2000, 67)])
def test_columns_of_many_tiles(torch_cuda, prec, n, cols):
    """Tiles on all XCDs, a last one in part, row pitches off the line size."""
    for pitch in (cols, cols + 3):
        x = rng.complex_normal(n + pitch, n * pitch).astype(CPLX_NP[prec]).reshape(n, pitch)
        plan = P.Plan("c2c", n, -1, prec, cols, pitch, 1, pitch, 1)
        assert "flex_c2c" in plan.describe() and "lanes" in plan.describe()
        y = to_dev(torch_cuda, np.full((n, pitch), 3 + 4j, CPLX_NP[prec]))
        plan.execute(to_dev(torch_cuda, x), y)
        y = from_dev(torch_cuda, y)
        assert relerr(y[:, :cols], np.fft.fft(x[:, :cols].astype(complex), axis=0)) < TOL[prec]
        assert np.all(y[:, cols:] == 3 + 4j)


@PRECS
@pytest.mark.parametrize("n", [64, 128])
def test_large_batch_of_short_reals(torch_cuda, prec, n):
    """64 MiB and more on both sides together, a last block in part."""
    m = n // 2 + 1
    hm = (1 << 26) // ((2 * n + 2) * np.dtype(REAL[prec]).itemsize) + 3
    x = rng.normal_f64(n, hm * n).astype(REAL[prec]).reshape(hm, n)
    ref = np.fft.rfft(x.astype(np.float64))
    y = to_dev(torch_cuda, np.zeros((hm, m), CPLX_NP[prec]))
    P.Plan("r2c", n, -1, prec, howmany=hm).execute(to_dev(torch_cuda, x), y)
    y = from_dev(torch_cuda, y)
    assert relerr(y, ref) < TOL[prec] and relerr(y[-40:], ref[-40:]) < TOL[prec]
    z = to_dev(torch_cuda, np.zeros((hm, n), REAL[prec]))
    P.Plan("c2r", n, 1, prec, howmany=hm).execute(to_dev(torch_cuda, ref.astype(CPLX_NP[prec])), z)
    z = from_dev(torch_cuda, z) / n
    assert relerr(z, x) < TOL[prec] and relerr(z[-40:], x[-40:]) < TOL[prec]
