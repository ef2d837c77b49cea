"""PlanFunction's output and gradient buffers: every element of a layout without
gaps is written (the allocator's memory holds NaN before), gaps are zero.

Tolerances are the suite's: relative L2 of 2e-6 (FP32), 1e-13 (FP64).
"""
import numpy as np
import pytest

import plfft_amd as P
from plfft_amd.autograd import PlanFunction, input_size, output_size
from gpu_util import TOL

pytestmark = pytest.mark.gpu

# kind, R2R kind, n, howmany, layout: packed, columns, gaps, one strided member
KINDS = [("c2c", 0), ("r2c", 0), ("c2r", 0), ("r2r", "dct2"), ("r2r", "dst2"), ("r2r", "dct3")]
LAYOUTS = ["packed", "columns", "gaps", "one", "longer"]


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("kind,r2r", KINDS)
@pytest.mark.parametrize("layout", LAYOUTS)
def test_buffers_written_or_zero(torch_cuda, prec, kind, r2r, layout):
    torch = torch_cuda
    for n, hm in ((12, 5), (64, 65), (1000, 3)):
        ic = n // 2 + 1 if kind == "c2r" else n
        oc = n // 2 + 1 if kind == "r2c" else n
        if layout == "one":
            hm, lay = 1, dict(istride=2, idist=0, ostride=3, odist=0)
        elif layout == "columns":
            lay = dict(istride=hm, idist=1, ostride=hm, odist=1)
        elif layout == "gaps":
            lay = dict(istride=2, idist=2 * ic + 3, ostride=1, odist=oc + 2)
        else:
            lay = dict(istride=1, idist=ic, ostride=1, odist=oc)
        plan = P.Plan(kind, n, 1 if kind == "c2r" else -1, prec, howmany=hm, r2r=r2r, **lay)
        real = torch.float32 if prec == "f32" else torch.float64
        cplx = torch.complex64 if prec == "f32" else torch.complex128
        xt = cplx if kind in ("c2c", "c2r") else real
        extra = 7 if layout == "longer" else 0  # an input buffer beyond the layout
        x = torch.randn(input_size(plan) + extra, dtype=xt, device="cuda", requires_grad=True)
        # what the allocator hands out next holds NaN
        junk = [torch.full((s,), float("nan"), dtype=t, device="cuda")
                for s in (output_size(plan), input_size(plan) + extra) for t in (real, cplx)]
        del junk
        y = PlanFunction.apply(x, plan)
        gy = torch.randn_like(y)
        (gx,) = torch.autograd.grad(y, x, gy)
        at = lambda c, s, d: (np.arange(hm)[:, None] * d + np.arange(c) * s).ravel()
        for buf, hit in ((y, at(oc, lay["ostride"], lay["odist"])),
                         (gx, at(ic, lay["istride"], lay["idist"]))):
            b = buf.detach().cpu().numpy()
            rest = np.ones(b.size, bool)
            rest[hit] = False
            assert np.all(np.isfinite(b)) and np.all(b[rest] == 0)
        # the gradient is the adjoint: <plan(d), gy> = <d, gx>
        d = torch.randn_like(x)
        z = PlanFunction.apply(d, plan)
        dot = lambda a, b: float((a.detach().to(torch.complex128).conj() *
                                  b.detach().to(torch.complex128)).sum().real)
        scale = float(z.detach().abs().double().norm() * gy.abs().double().norm())
        assert abs(dot(z, gy) - dot(d, gx)) < TOL[prec] * scale
