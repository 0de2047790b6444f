"""GPU tests of the main loop on small lattices, whose pairs of steps run as
single steps in smaller blocks: grids around each block size (64 threads up to
512, with and without a remainder), FP64, bit for bit against the oracle; the
per-call pairing with the sweep asked for, which such lattices no longer take
by themselves; and the sweep along z slabs of every residue modulo a wave,
bit for bit against single steps."""
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
    c.macrovar()


# nodes: 2 (one lane pair), 63, 64 blocks of 64, 256 blocks of 64, one block
# more, 128-, 256- and 512-thread blocks with a remainder
@pytest.mark.parametrize("lx,ly,lz", [(2, 1, 1), (3, 7, 3), (16, 16, 16), (16, 32, 32), (17, 31, 32), (33, 31, 31),
                                      (32, 32, 33), (47, 40, 33), (64, 64, 32), (65, 64, 33)])
def test_steps_at_every_block_size(lx, ly, lz):
    u = workloads.laminar_parabola_noise(lx, ly, lz, seed=8)
    ref = O.OracleChannel(lx, ly, lz)
    _start(ref, u)
    with d3q19.Channel(lx, ly, lz) as ch:
        _start(ch, u)
        ref.run(3)
        ch.run(3)
        ref.run_forcingp(3, 3, 6)  # two perturbed steps, one uniform
        ch.run_forcingp(3, 3, 6)
        assert np.array_equal(bits(ch.download_f()), bits(ref.f))
        ref.rhoupdat()  # a step with stored fields
        ch.rhoupdat()
        ref.collision_MRT()
        ch.collision_MRT()
        assert np.array_equal(bits(ch.download_f()), bits(ref.f))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_per_call_pairs_with_the_sweep_asked_for(monkeypatch, prec):
    u = workloads.laminar_parabola_noise(24, 20, 18, seed=9)
    monkeypatch.setenv("LBM_BLOCK_PLANES", "5")
    paired = d3q19.Channel(24, 20, 18, prec)
    monkeypatch.delenv("LBM_BLOCK_PLANES")
    single = d3q19.Channel(24, 20, 18, prec)
    with paired, single:
        for c in (paired, single):
            _start(c, u)
            for k in range(9):
                c.collision_MRT()
                c.macrovar()
                if k == 4:
                    c.stats_accumulate()  # launches what is deferred
        assert np.array_equal(bits(paired.download_post()), bits(single.download_post()))
        assert np.array_equal(bits(paired.statistc2()), bits(single.statistc2()))


# lx * ly modulo 64: 0, 1, 32, 63 and others; slabs below a wave and of several
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("lx,ly,lz,k", [(16, 8, 9, 3), (5, 13, 11, 2), (12, 8, 7, 3), (7, 9, 12, 4), (3, 7, 5, 5),
                                        (13, 11, 10, 1), (33, 31, 17, 6), (9, 7, 1, 1), (9, 7, 2, 2)])
def test_sweep_of_slabs_that_do_not_fill_waves(monkeypatch, prec, lx, ly, lz, k):
    u = workloads.laminar_parabola_noise(lx, ly, lz, seed=10)
    monkeypatch.setenv("LBM_BLOCK_AXIS", "z")
    monkeypatch.setenv("LBM_BLOCK_PLANES", str(k))
    swept = d3q19.Channel(lx, ly, lz, prec)
    monkeypatch.setenv("LBM_BLOCK_PLANES", "0")
    single = d3q19.Channel(lx, ly, lz, prec)
    with swept, single:
        for c in (swept, single):
            _start(c, u)
            c.run(6)
            c.run_forcingp(6, 4, 9)
        a, b = swept.download_post(), single.download_post()
    if prec == "fp64":
        assert np.array_equal(bits(a), bits(b))
    else:  # FMA contraction may differ between the kernels: an ulp of the largest value
        assert np.max(np.abs(a - b)) <= 1e-6 * np.max(np.abs(b))
