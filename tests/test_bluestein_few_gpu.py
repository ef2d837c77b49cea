"""Bluestein in FP64 on either side of the line between few members (8 points a
thread) and many (16), against numpy's FP64 transform. Tolerance: the suite's."""
import numpy as np
import pytest

import plfft_amd as P
from plfft_amd import rng
from gpu_util import TOL, from_dev, relerr, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,few,many", [(58, "r8x2x8_t16", "r16x8_t8"), (458, "r8x2x8x8_t128", "r16x4x16_t64"),
                                        (838, "r8x4x8x8_t256", "r16x8x16_t128")])
def test_few_and_many_members(torch_cuda, n, few, many):
    for hm, chain in ((1, few), (17, few), (6003, many)):
        x = rng.complex_normal(n + hm, hm * n).reshape(hm, n)
        for direction, f in ((-1, np.fft.fft), (1, np.fft.ifft)):
            plan = P.Plan("c2c", n, direction, "f64", howmany=hm)
            assert chain in plan.describe()
            y = to_dev(torch_cuda, np.zeros((hm, n), complex))
            plan.execute(to_dev(torch_cuda, x), y)
            ref = f(x) * (n if direction > 0 else 1)
            assert relerr(from_dev(torch_cuda, y), ref) < TOL["f64"], plan.describe()
