"""GPU tests of the coupled particle loop, whose classification runs beside
the collision: against the oracle (FP64, bit for bit) at radii on both sides of
the largest box whose node flags are staged in LDS, over several calls; and
against the routines called one by one, with the link lists, for overlapping
spheres, spheres that run into each other, and a loop entered without macrovar."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads
import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


def _start(ch, seed):
    ux, uy, uz = workloads.laminar_parabola_noise(ch.lx, ch.ly, ch.lz, seed=seed)
    ch.set_macros(ux=ux, uy=uy, uz=uz)
    ch.FORCING()
    ch.initpop()
    ch.macrovar()


# links: (2 R + 6)^3 flags staged up to 16 384, R = 9.7; uncovering: (2 R + 3)^3, R = 11.2
@pytest.mark.parametrize("rad", [9.2, 9.7, 10.4, 11.3, 12.6])
def test_radii_around_the_staging_limit(rad):
    lx, ly, lz = 64, 44, 40
    pos = np.array([[17.3, 5.2, 33.9], [45.7, 25.0, 11.5]])
    vel = np.array([[0.0, 0.3, -0.2], [0.1, -0.2, 0.25]])
    p = d3q19.para(lx, laminar=True)
    with d3q19.Channel(lx, ly, lz, params=p) as ch:
        _start(ch, 2)
        L0 = ch.download_post()
        ch.particles_create(pos, vel=vel, rad=rad, nave=2)
        g = O.particle_geometry(lx, ly, lz, len(pos), rad, force=(0.0, p["force_in_y"], 0.0))
        ref = O.OracleParticleChannel(O.para(lx, ly, lz, laminar=True), g, L0, pos, vel=vel)
        for first, n in ((0, 1), (1, 3), (4, 2)):
            ch.run_particles(n, istep0=first)
            ref.step(n, istep0=first, nave=2)
        got = ch.particles_get()
        assert np.array_equal(ch.particles_solid(), ref.solid)
        assert np.array_equal(bits(got["pos"].reshape(-1)), bits(ref.X))
        assert np.array_equal(bits(got["vel"].reshape(-1)), bits(ref.V))
        fluid = np.flatnonzero(ref.solid < 0)
        assert np.array_equal(bits(ch.download_post()[:, fluid]), bits(ref.post.reshape(19, -1)[:, fluid]))


def _by_calls(ch, n):
    for _ in range(n):
        ch.beads_collision()
        ch.beads_move()
        ch.collision_MRT()
        ch.macrovar()
        ch.beads_links()
        ch.beads_filling()


def _state(ch):
    out = ch.particles_get()
    out["solid"] = ch.particles_solid()
    cap, out["counts"], node, dirs, q = ch.particles_links()
    valid = (np.arange(cap)[None, :] < out["counts"][:, None]).ravel()
    out["node"], out["dirs"], out["q"] = node[valid], dirs[valid], q[valid]
    out["post"] = ch.download_post()
    out["fields"] = np.stack(ch.macrovar(download=True))
    return out


@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("pos,vel", [
    ([[12.0, 9.0, 9.0], [16.0, 12.0, 10.0]], [[0.3, 0.2, 0.0], [-0.3, -0.2, 0.1]]),      # overlap, moving into each other
    ([[16.0, 12.0, 10.0], [12.0, 9.0, 9.0]], [[-0.4, 0.0, 0.1], [0.4, 0.3, 0.0]]),      # the other id wins
    ([[8.0, 0.5, 17.5], [8.4, 9.6, 17.0], [20.0, 18.0, 2.0]], [[0.0, 0.5, 0.0]] * 3),     # across the period
])
@pytest.mark.parametrize("enter", ["macrovar", "collision"])
def test_equals_the_calls_one_by_one(prec, pos, vel, enter):
    with d3q19.Channel(28, 20, 18, prec, laminar=True) as a, d3q19.Channel(28, 20, 18, prec, laminar=True) as b:
        for ch in (a, b):
            _start(ch, 3)
            ch.particles_create(np.array(pos), vel=np.array(vel), rad=4.6, visc=0.1)
            if enter == "collision":  # the loop's first step then makes the fields of the lattice before
                ch.beads_collision()
                ch.collision_MRT()
        a.run_particles(3)
        a.run_particles(4, istep0=3)
        _by_calls(b, 7)
        sa, sb = _state(a), _state(b)
    # the overlaps are violent enough for FP32 and FP16 populations to leave
    # their range within seven steps: a NaN equals a NaN here
    for k in sb:
        assert np.array_equal(sa[k], sb[k], equal_nan=True), k
