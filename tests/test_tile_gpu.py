"""The tile kernels (columns of a matrix; four-step with a blocked workspace)
against the FP64 oracle, at the edges of their tiles and over the layouts
that the planner hands them.

Tolerances are the suite's: relative L2 of 2e-6 (FP32 arithmetic), 1e-13
(FP64), and the storage rounding of f16 / bf16.
"""
import numpy as np
import pytest

import plfft_amd as P
from plfft_amd import rng
from gpu_util import CPLX_NP, TOL, bf16_bits, bf16_to_f32, from_dev, relerr, to_dev

pytestmark = pytest.mark.gpu

# columns enough for 64 tiles of the widest kernel of each length (fewer keep
# the general kernel)
MEMBERS = {64: 4096, 128: 2048, 256: 2048, 512: 2048, 1024: 1024, 2048: 1024}
COLS = [("f32", n) for n in (64, 128, 256, 512, 1024, 2048)] + \
       [("f64", n) for n in (64, 128, 256, 512, 1024)] + \
       [("f16", n) for n in (64, 128, 256, 512, 1024)] + [("bf16", 256)]


def _store(torch, z, prec):
    """complex128 host array -> device buffer of the storage type."""
    if prec in CPLX_NP and prec != "f16":
        return to_dev(torch, z.astype(CPLX_NP[prec]))
    r = np.ascontiguousarray(z.astype(np.complex64)).view(np.float32)
    if prec == "f16":
        return to_dev(torch, r.astype(np.float16))
    return to_dev(torch, bf16_bits(r).view(np.int16))


def _load(torch, d, prec):
    a = from_dev(torch, d)
    if prec in ("f32", "f64"):
        return a.astype(np.complex128)
    r = a.astype(np.float32) if prec == "f16" else bf16_to_f32(a.view(np.uint16))
    return r.astype(np.float64).view(np.complex128)


def _signal(seed, count, prec):
    x = rng.complex_normal(seed, count)
    if prec in ("f32", "f64"):
        return x.astype(CPLX_NP[prec]).astype(np.complex128)
    r = np.ascontiguousarray(x).view(np.float64).astype(np.float32)
    r = r.astype(np.float16).astype(np.float32) if prec == "f16" else bf16_to_f32(bf16_bits(r))
    return r.astype(np.float64).view(np.complex128)


@pytest.mark.parametrize("prec,n", COLS)
def test_columns_vs_oracle(torch_cuda, orc, prec, n):
    """Whole tiles, a remainder of one member, row pitches off the line size,
    padded rows and members two elements apart; both directions, in place."""
    torch = torch_cuda
    m = MEMBERS[n]
    for hm, gap, dist in ((m, 0, 1), (m + 1, 0, 1), (m + 13, 3, 1), (m + 6, 0, 2)):
        st = hm * dist + gap
        size = n * st
        x = _signal(n + hm, size, prec)
        for direction in (-1, 1) if gap else (1,):
            plan = P.Plan("c2c", n, direction, prec, hm, st, dist, st, dist, may_alias=True)
            assert "tile_c2c" in plan.describe()
            d = _store(torch, x, prec)
            y0 = _store(torch, np.full(size, 3 + 4j), prec)
            plan.execute(d, y0)
            ref = orc.c2c_batched(x, n, direction, hm, st, dist, st, dist, size)
            hit = (np.arange(n)[:, None] * st + np.arange(hm) * dist).ravel()
            y = _load(torch, y0, prec)
            assert relerr(y[hit], ref[hit]) < TOL[prec], plan.describe()
            rest = np.ones(size, bool)
            rest[hit] = False
            assert np.all(y[rest] == 3 + 4j)  # the gaps are not written
            plan.execute(d, d)
            assert np.array_equal(_load(torch, d, prec)[hit], y[hit])


def test_columns_rule():
    """Few columns, packed members and transposing layouts keep the general
    kernels."""
    n = 1024
    def d(*a):
        return P.Plan("c2c", n, -1, "f32", *a).describe()
    assert "tile_c2c" in d(4096, 4096, 1, 4096, 1)
    assert "tile_c2c" not in d(16, 16, 1, 16, 1)
    assert "tile_c2c" not in d(4096, 1, n, 1, n)
    assert "tile_c2c" not in d(4096, 4096, 1, 1, n)


FOURSTEP = [("f32", 16), ("f32", 17), ("f32", 18), ("f32", 19), ("f32", 20), ("f32", 21),
            ("f32", 22), ("f64", 15), ("f64", 16), ("f64", 17), ("f64", 18), ("f64", 19),
            ("f64", 20), ("f64", 21), ("f64", 22), ("f16", 16), ("f16", 17), ("f16", 18),
            ("f16", 19), ("f16", 20), ("bf16", 16)]


@pytest.mark.parametrize("prec,lg", FOURSTEP)
def test_fourstep_vs_oracle(torch_cuda, orc, prec, lg):
    """Packed members, members off the line boundaries and (short lengths)
    strided sides, in both directions."""
    torch = torch_cuda
    n = 1 << lg
    hm = max(4, (1 << 22) >> lg) if prec in ("f32", "f64") else 2  # a block per CU
    layouts = [(hm, 1, n, 1, n)]
    if lg <= 18:
        layouts += [(hm + 1, 1, n + 1, 1, n + 3), (hm, 2, 2 * n + 1, 3, 3 * n)]
    for i, (hm, is_, id_, os_, od_) in enumerate(layouts):
        isz = (hm - 1) * id_ + (n - 1) * is_ + 1
        osz = (hm - 1) * od_ + (n - 1) * os_ + 1
        x = _signal(lg + i, isz, prec)
        d = _store(torch, x, prec)
        for direction in (-1, 1) if i == 0 else (1,):
            plan = P.Plan("c2c", n, direction, prec, hm, is_, id_, os_, od_)
            assert "tile_col" in plan.describe() and "tile_row" in plan.describe()
            y0 = _store(torch, np.full(osz, 3 + 4j), prec)
            plan.execute(d, y0)
            y = _load(torch, y0, prec)
            ref = orc.c2c_batched(x, n, direction, hm, is_, id_, os_, od_, osz)
            hit = (np.arange(hm)[:, None] * od_ + np.arange(n) * os_).ravel()
            assert relerr(y[hit], ref[hit]) < TOL[prec], plan.describe()
            rest = np.ones(osz, bool)
            rest[hit] = False
            assert np.all(y[rest] == 3 + 4j)
