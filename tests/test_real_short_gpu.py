"""R2C / C2R of short packed members, which pass through LDS a block at a time:
one member, whole blocks and one more or less, beside layouts with a gap (the
strided path of the same kernels); and C2R bins 0 and n/2, which count as real
whatever their imaginary parts hold, NaN included.

Tolerances are the suite's: relative L2 of 2e-6 (FP32), 1e-13 (FP64).
"""
import numpy as np
import pytest

import plfft_amd as P
from plfft_amd import rng
from gpu_util import TOL, from_dev, relerr, to_dev

pytestmark = pytest.mark.gpu

REAL = {"f32": np.float32, "f64": np.float64}
CPLX = {"f32": np.complex64, "f64": np.complex128}


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("n", [64, 128])
def test_short_r2c_c2r(torch_cuda, prec, n):
    m, torch = n // 2 + 1, torch_cuda
    for hm in (1, 31, 32, 33, 63, 64, 65, 200):
        for gap in (0, 2):
            nr, nc = n + gap, m + gap
            x = rng.complex_normal(n + hm, hm * nr).real.astype(REAL[prec]).reshape(hm, nr)
            F = rng.complex_normal(1000 + n + hm, hm * nc).astype(CPLX[prec]).reshape(hm, nc)
            y = to_dev(torch, np.full((hm, nc), 3 + 4j, CPLX[prec]))
            z = to_dev(torch, np.full((hm, nr), 5, REAL[prec]))
            P.Plan("r2c", n, -1, prec, howmany=hm, idist=nr, odist=nc).execute(to_dev(torch, x), y)
            P.Plan("c2r", n, 1, prec, howmany=hm, idist=nc, odist=nr).execute(to_dev(torch, F), z)
            y, z = from_dev(torch, y), from_dev(torch, z)
            G = F[:, :m].astype(complex)
            G[:, 0].imag = G[:, -1].imag = 0
            ref = np.fft.irfft(G, n=n) * n
            assert relerr(y[:, :m].ravel(), np.fft.rfft(x[:, :n].astype(float)).ravel()) < TOL[prec]
            assert relerr(z[:, :n].ravel(), ref.ravel()) < TOL[prec]
            assert np.all(y[:, m:] == 3 + 4j) and np.all(z[:, n:] == 5)


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("n", [16, 64, 100, 1000])
def test_c2r_ignores_imaginary_of_real_bins(torch_cuda, prec, n):
    torch, m = torch_cuda, n // 2 + 1
    F = rng.complex_normal(n, 3 * m).astype(CPLX[prec]).reshape(3, m)
    F[:, 0].imag = F[:, -1].imag = 0
    plan = P.Plan("c2r", n, 1, prec, howmany=3)
    out = []
    for im in (0, np.nan, np.inf):
        G = F.copy()
        G.imag[:, 0] = G.imag[:, -1] = im
        z = to_dev(torch, np.zeros((3, n), REAL[prec]))
        plan.execute(to_dev(torch, G), z)
        out.append(from_dev(torch, z))
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
    assert relerr(out[0].ravel(), (np.fft.irfft(F.astype(complex), n=n) * n).ravel()) < TOL[prec]
