"""Convolution kernels on the two-transform tile engine (one-block Bluestein of
a compile-time padded length; the row pass of three-pass chirp-z and Rader)
against an FP64 DFT: the shortest and longest length of every padded length,
every row length, partial last blocks, strides, both directions.

Tolerances are the suite's: relative L2 of 2e-6 (FP32 arithmetic), 1e-13
(FP64), and the storage rounding of f16 / bf16.
"""
import numpy as np
import pytest

import plfft_amd as P
from gpu_util import TOL, relerr
from test_mixed_gpu import TOL_MIX
from test_tile_gpu import _load, _signal, _store

pytestmark = pytest.mark.gpu

BLUE = [(p, 1 << k) for p in ("f32", "f64", "f16", "bf16")
        for k in range(7, 13 if p == "f64" else 15)]
# 2 * prime and the like, just below half of M = n1 * n2 (rows of n2 points)
CZ = [("f32", n) for n in (8198, 12278, 16382, 24574, 32762, 49150, 65534, 98302, 131066, 196606,
                           400018)] + \
     [("f64", n) for n in (2062, 4094, 4106, 8198, 12278, 16382, 24574, 65534, 131066)] + \
     [("f16", 16382), ("bf16", 24574)]
RADER = [("f32", 65537), ("f32", 786433), ("f64", 12289), ("f64", 65537), ("f16", 65537)]


def _dft(x, direction):
    return np.fft.fft(x) if direction < 0 else np.fft.ifft(x) * x.shape[-1]


def _check(torch, prec, n, cases, what, tol):
    for hm, is_, id_, os_, od_ in cases:
        isz, osz = (hm - 1) * id_ + (n - 1) * is_ + 1, (hm - 1) * od_ + (n - 1) * os_ + 1
        x = _signal(n + hm, isz, prec)
        rows = np.arange(hm)[:, None] * id_ + np.arange(n) * is_
        hit = np.arange(hm)[:, None] * od_ + np.arange(n) * os_
        for direction in (-1, 1):
            plan = P.Plan("c2c", n, direction, prec, hm, is_, id_, os_, od_)
            assert what in plan.describe()
            d = _store(torch, x, prec)
            o = _store(torch, np.full(osz, 3 + 4j), prec)
            plan.execute(d, o)
            y = _load(torch, o, prec)
            assert relerr(y[hit].ravel(), _dft(x[rows], direction).ravel()) < tol, plan.describe()
            rest = np.ones(osz, bool)
            rest[hit.ravel()] = False
            assert np.all(y[rest] == 3 + 4j)  # the gaps are not written


@pytest.mark.parametrize("prec,M", BLUE)
def test_bluestein(torch_cuda, prec, M):
    tag = f" M={M} "
    span = range(M // 4 + 2, M // 2 + 2)
    found = 0
    for order in (span, reversed(span)):  # the shortest and the longest length
        n = next((n for n in order
                  if f"(bluestein n={n}{tag}" in P.Plan("c2c", n, -1, prec).describe()), None)
        if n is None:
            continue
        found += 1
        hm = max(3, 2000 // n) + 1
        _check(torch_cuda, prec, n, [(hm, 1, n, 1, n), (3, 2, 2 * n + 3, 3, 3 * n + 1)],
               tag, TOL[prec])
    assert found


@pytest.mark.parametrize("prec,n", CZ)
def test_chirpz_rows(torch_cuda, prec, n):
    # FP64 padded lengths to 8192 fit one block of the runtime chain
    what = "bluestein" if prec == "f64" and n < 4097 else "chirpz3"
    _check(torch_cuda, prec, n, [(3, 1, n, 1, n), (2, 2, 2 * n + 3, 1, n + 5)], what, TOL[prec])


@pytest.mark.parametrize("prec,n", RADER)
def test_rader_rows(torch_cuda, prec, n):
    _check(torch_cuda, prec, n, [(2, 1, n, 1, n), (3, 1, n + 2, 2, 2 * n)], "rader3", TOL[prec])


@pytest.mark.parametrize("prec", ["f32", "f64", "f16"])
def test_mixed_groups(torch_cuda, prec):
    """Gathered members of every padded length, in groups of one and of many."""
    torch = torch_cuda
    lengths = [29, 37, 67, 131, 263, 521, 1031, 1999, 2049 * 2, 2111, 3079, 4099, 6151, 8209, 12301,
               16411, 24593, 32771] + [59, 97, 1031, 3079] * 9 + [2 * 4099, 31 * 37 * 2]
    x = _signal(5, sum(lengths), prec)
    for direction in (-1, 1):
        plan = P.MixedPlan(lengths, direction, prec)
        d = _store(torch, x, prec)
        o = _store(torch, np.zeros(x.size, complex), prec)
        plan.execute(d, o)
        y = _load(torch, o, prec)
        at = 0
        for n in lengths:
            ref = _dft(x[at:at + n], direction)
            assert relerr(y[at:at + n], ref) < TOL_MIX[prec], (n, direction)
            at += n
