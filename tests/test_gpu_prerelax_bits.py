"""GPU test of the pre-relaxation loop against rhoupdat and collision_MRT called
one by one, bit for bit in every precision: changes, populations and fields, on
lattices that the step takes every way through the caches."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16", "fp16c"])
@pytest.mark.parametrize("lx,ly,lz", [(2, 3, 1), (16, 16, 8), (48, 50, 50), (61, 79, 79), (97, 97, 97), (130, 130, 130)])
def test_equals_the_calls_bit_for_bit(prec, lx, ly, lz):
    u = workloads.laminar_parabola_noise(lx, ly, lz, seed=4)
    with d3q19.Channel(lx, ly, lz, prec) as a, d3q19.Channel(lx, ly, lz, prec) as b:
        for c in (a, b):
            c.FORCING()
            c.set_macros(ux=u[0], uy=u[1], uz=u[2])
            c.initpop()
        for n in (1, 2, 6):
            it, err = a.prerelax(-1.0, n - 2)
            assert it == n - 1
            for _ in range(n):
                err_b = b.rhoupdat()
                b.collision_MRT()
            assert err == err_b
            assert np.array_equal(a.download_post(), b.download_post())
        fa, fb = a.macrovar(download=True), b.macrovar(download=True)
        assert all(np.array_equal(x, y) for x, y in zip(fa, fb))
