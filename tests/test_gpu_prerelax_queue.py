"""GPU test of the pre-relaxation loop entered while the handle's stream still
works: rhoupdat calls that do not ask for their maximum (a null pointer, which
the C ABI allows) return before their kernels have run, and nothing they store
may be taken for an iteration's result."""
import ctypes

import numpy as np
import pytest

import d3q19
from d3q19 import workloads

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


def _start(lx, ly, lz, prec):
    ch = d3q19.Channel(lx, ly, lz, prec)
    u = workloads.laminar_parabola_noise(lx, ly, lz, seed=6)
    ch.set_macros(ux=u[0], uy=u[1], uz=u[2])
    ch.FORCING()
    ch.initpop()
    return ch


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_maxima_queued_before_the_loop_are_not_its_results(prec):
    lx, ly, lz, queued, n = 130, 130, 130, 200, 5
    lib = d3q19.load_library()
    with _start(lx, ly, lz, prec) as b:  # call by call, waiting for every maximum
        b.rhoupdat()
        b.collision_MRT()
        want = []
        for _ in range(n):
            want.append(b.rhoupdat())
            b.collision_MRT()
        fb = b.download_f()
    assert min(want) > 0.0
    with _start(lx, ly, lz, prec) as a:
        # from the second of these on nothing changes: maxima of 0, below any limit
        for _ in range(queued):
            assert lib.lbm_rhoupdat(a._h, None) == 0
        a.collision_MRT()
        errs, done = np.full(n, -1.0), ctypes.c_int(-1)
        rc = lib.lbm_prerelax(a._h, 0.5 * min(want), n, ctypes.byref(done), errs.ctypes.data_as(ctypes.c_void_p))
        assert rc == 0, lib.lbm_last_error()
        assert done.value == n, errs
        fa = a.download_f()
    if prec == "fp64":
        assert errs.tolist() == want
        assert np.array_equal(bits(fa), bits(fb))
    else:
        # an ulp of the largest value per population from contraction
        tol = 2.0 ** -20 * np.max(np.abs(fb))
        assert np.max(np.abs(errs - want)) <= 19.0 * tol
        assert np.max(np.abs(fa - fb)) <= tol
