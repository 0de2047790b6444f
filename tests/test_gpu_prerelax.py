"""GPU tests of the pre-relaxation loop, whose iterations are one pass each and
run ahead of the host's test of the density change: number of iterations, last
change and populations against the oracle (FP64, bit for bit) and against the
two routines called one by one (FP32; a force that varies over the nodes)."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads
import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


def _start(c, u):
    c.FORCING()
    if isinstance(c, O.OracleChannel):
        c.ux[:], c.uy[:], c.uz[:] = u
    else:
        c.set_macros(ux=u[0], uy=u[1], uz=u[2])
    c.initpop()


def _by_calls(ch, iterations):
    for _ in range(iterations):
        err = ch.rhoupdat()
        ch.collision_MRT()
    return err


# `last`: the iteration whose change ends the loop (the first, one of those run
# ahead, the last and the first of a group of 64) or, with None, maxiter does
@pytest.mark.parametrize("lx,ly,lz", [(2, 1, 1), (7, 5, 3), (16, 12, 8), (17, 31, 33)])
@pytest.mark.parametrize("last,maxiter", [(0, 100), (1, 100), (3, 100), (4, 100), (63, 100), (64, 100),
                                          (None, -1), (None, 0), (None, 3), (None, 62), (None, 63), (None, 70)])
def test_ends_where_the_oracle_ends(lx, ly, lz, last, maxiter):
    u = workloads.laminar_parabola_noise(lx, ly, lz, seed=3)
    ref = O.OracleChannel(lx, ly, lz)
    _start(ref, u)
    eps = -1.0
    if last is not None:  # the change of iteration `last`, if none before is smaller
        errs = []
        for _ in range(last + 1):
            old = ref.rho.copy()
            ref.rhoupdat()
            errs.append(float(np.max(np.abs(ref.rho - old))))
            ref.collision_MRT()
        eps = errs[-1]
        ref = O.OracleChannel(lx, ly, lz)
        _start(ref, u)
    want = ref.prerelax(eps, maxiter)
    with d3q19.Channel(lx, ly, lz) as ch:
        _start(ch, u)
        assert ch.prerelax(eps, maxiter) == want
        assert np.array_equal(bits(ch.download_f()), bits(ref.f))
        ref.rhoupdat()  # the loop leaves rho and the lattices as the calls do
        ch.rhoupdat()
        ref.collision_MRT()
        ch.collision_MRT()
        ref.macrovar()
        ch.macrovar()
        ref.run(3)
        ch.run(3)
        assert np.array_equal(bits(ch.download_f()), bits(ref.f))


# one lattice of 0.3, 18, 58, 138 and 335 MB in FP64, half that in FP32: every
# way of a step through the caches
@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("lx,ly,lz", [(16, 16, 8), (48, 50, 50), (61, 79, 79), (97, 97, 97), (130, 130, 130)])
def test_equals_the_calls_one_by_one(prec, lx, ly, lz):
    u = workloads.laminar_parabola_noise(lx, ly, lz, seed=4)
    with d3q19.Channel(lx, ly, lz, prec) as a, d3q19.Channel(lx, ly, lz, prec) as b:
        for c in (a, b):
            _start(c, u)
        it, err = a.prerelax(-1.0, 5)
        err_b = _by_calls(b, 7)
        assert it == 6
        fa, fb = a.download_f(), b.download_f()
        assert np.array_equal(bits(a.macrovar(download=True)[0]), bits(b.macrovar(download=True)[0])) or prec != "fp64"
    top = np.max(np.abs(fb))
    # the same arithmetic; FMA contraction may differ between the kernels, which
    # moves a value by an ulp of the largest one
    tol = {"fp64": 0.0, "fp32": 2.0 ** -20, "fp16": 2.0 ** -9}[prec] * top
    assert np.max(np.abs(fa - fb)) <= tol
    assert abs(err - err_b) <= 19.0 * tol


def test_force_that_varies_over_the_nodes():
    u = workloads.laminar_parabola_noise(24, 20, 18, seed=5)
    with d3q19.Channel(24, 20, 18) as a, d3q19.Channel(24, 20, 18) as b:
        for c in (a, b):
            _start(c, u)
            c.FORCINGP(7)
        assert a.prerelax(-1.0, 66) == (67, _by_calls(b, 68))
        assert np.array_equal(bits(a.download_f()), bits(b.download_f()))
