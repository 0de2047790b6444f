"""GPU tests of the coupled particle loop in both of its forms, on one stream and
with the particle work on a second stream beside the collision (the form of
lattices above 260 MB), whichever the lattice's size: against the oracle (FP64,
bit for bit) at box edges, radii around the limit of the node flags staged in
LDS and long refill lists, with the link lists; against the routines called one
by one, entered with and without macrovar; and one lattice above the limit."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads
import oracle as O
from test_gpu_particle_overlap import _by_calls, _start, _state, bits

pytestmark = pytest.mark.gpu


@pytest.fixture(params=["1", "2"])
def streams(request, monkeypatch):
    monkeypatch.setenv("LBM_PART_STREAMS", request.param)
    return request.param


def test_values_of_the_switch(monkeypatch):
    for bad in ("0", "3", "", "two"):
        monkeypatch.setenv("LBM_PART_STREAMS", bad)
        with pytest.raises(d3q19.LbmError, match="LBM_PART_STREAMS"):
            d3q19.Channel(12, 10, 6)


@pytest.mark.parametrize("lx,ly,lz,rad,pos,vel", [
    (24, 20, 18, 1.5, [[4.2, 0.3, 17.8], [12.0, 10.0, 9.0]], 0.05),    # boxes below a block's threads, wrapping
    (24, 20, 18, 3.6, [[4.0, 19.7, 0.2], [17.1, 8.3, 9.4]], 0.2),      # near the wall
    (40, 14, 13, 5.0, [[11.3, 6.5, 6.1]], 0.1),                        # as wide as both periods
    (64, 48, 40, 9.0, [[14.5, 3.2, 37.9], [42.3, 24.0, 15.5]], 0.3),   # several passes, long refill lists
    (64, 44, 40, 9.7, [[17.3, 5.2, 33.9], [45.7, 25.0, 11.5]], 0.3),   # (2 R + 6)^3 just staged
    (64, 44, 40, 9.9, [[17.3, 5.2, 33.9], [45.7, 25.0, 11.5]], 0.3),   # links from memory, uncovering staged
    (64, 44, 40, 12.6, [[17.3, 5.2, 33.9], [45.7, 25.0, 11.5]], 0.3),  # both from memory
])
def test_coupled_steps_equal_the_oracle(streams, lx, ly, lz, rad, pos, vel):
    pos = np.array(pos)
    v = np.zeros_like(pos)
    v[:, 1], v[:, 2] = vel, -0.7 * vel
    p = d3q19.para(lx, laminar=True)
    with d3q19.Channel(lx, ly, lz, params=p) as ch:
        _start(ch, 2)
        L0 = ch.download_post()
        ch.particles_create(pos, vel=v, rad=rad, nave=3)
        g = O.particle_geometry(lx, ly, lz, len(pos), rad, force=(0.0, p["force_in_y"], 0.0))
        ref = O.OracleParticleChannel(O.para(lx, ly, lz, laminar=True), g, L0, pos, vel=v)
        for first, n in ((0, 1), (1, 4), (5, 2)):
            ch.run_particles(n, istep0=first)
            ref.step(n, istep0=first, nave=3)
        got = ch.particles_get()
        assert np.array_equal(ch.particles_solid(), ref.solid)
        assert np.array_equal(bits(got["pos"].reshape(-1)), bits(ref.X))
        assert np.array_equal(bits(got["vel"].reshape(-1)), bits(ref.V))
        assert np.array_equal(bits(got["omg"].reshape(-1)), bits(ref.W))
        fluid = np.flatnonzero(ref.solid < 0)
        assert np.array_equal(bits(ch.download_post()[:, fluid]), bits(ref.post.reshape(19, -1)[:, fluid]))


@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("pos,vel", [
    ([[12.0, 9.0, 9.0], [16.0, 12.0, 10.0]], [[0.02, 0.01, 0.0], [-0.02, -0.01, 0.01]]),  # overlap
    ([[8.0, 0.5, 17.5], [8.4, 9.6, 17.0], [20.0, 18.0, 2.0]], [[0.0, 0.2, 0.0]] * 3),      # across the period
])
@pytest.mark.parametrize("enter", ["macrovar", "collision"])
def test_equals_the_calls_one_by_one(streams, prec, pos, vel, enter):
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
    for k in sb:
        assert np.array_equal(sa[k], sb[k], equal_nan=True), k


def test_lattice_above_the_limit_equals_the_calls(monkeypatch):
    """96x194x96 in FP64, 272 MB a lattice: two streams by the rule on sizes."""
    monkeypatch.delenv("LBM_PART_STREAMS", raising=False)
    lx, ly, lz = 96, 194, 96
    pos = workloads.sphere_positions(lx, ly, lz, 12, 5.3, seed=8)
    vel = np.tile([[0.03, 0.2, -0.1], [-0.02, -0.1, 0.2]], (6, 1))
    with d3q19.Channel(lx, ly, lz, laminar=True) as a, d3q19.Channel(lx, ly, lz, laminar=True) as b:
        for ch in (a, b):
            _start(ch, 3)
            ch.particles_create(pos, vel=vel, rad=5.3, visc=0.1)
        a.run_particles(6)
        _by_calls(b, 6)
        sa, sb = _state(a), _state(b)
    for k in sb:
        assert np.array_equal(sa[k], sb[k]), k
