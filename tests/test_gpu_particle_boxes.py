"""GPU test of the particle kernels at the edges of their work split, FP64
coupled steps bit for bit against the oracle: boxes of fewer nodes than a
block's threads and of several passes, boxes cut by a wall, boxes as wide as
a period, boxes that wrap around it, and spheres fast enough to uncover more
nodes than one pass of the refill's waves takes."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads
import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


@pytest.mark.parametrize("lx,ly,lz,rad,pos,vel", [
    (24, 20, 18, 1.5, [[4.2, 0.3, 17.8], [12.0, 10.0, 9.0]], 0.05),    # 5^3 nodes, wrapping in y and z
    (24, 20, 18, 3.6, [[4.0, 19.7, 0.2], [17.1, 8.3, 9.4]], 0.2),      # 9^3-10^3, near the wall
    (40, 14, 13, 5.0, [[11.3, 6.5, 6.1]], 0.1),                        # box as wide as both periods
    (64, 48, 40, 9.0, [[14.5, 3.2, 37.9], [42.3, 24.0, 15.5]], 0.3),   # several passes, long refill lists
])
def test_coupled_steps_at_box_edges(lx, ly, lz, rad, pos, vel):
    pos = np.array(pos)
    v = np.zeros_like(pos)
    v[:, 1], v[:, 2] = vel, -0.7 * vel
    p = d3q19.para(lx, laminar=True)
    ux, uy, uz = workloads.laminar_parabola_noise(lx, ly, lz, seed=2)
    with d3q19.Channel(lx, ly, lz, params=p) as ch:
        ch.set_macros(ux=ux, uy=uy, uz=uz)
        ch.FORCING()
        ch.initpop()
        ch.macrovar()
        L0 = ch.download_post()
        ch.particles_create(pos, vel=v, rad=rad, nave=3)
        g = O.particle_geometry(lx, ly, lz, len(pos), rad, force=(0.0, p["force_in_y"], 0.0))
        ref = O.OracleParticleChannel(O.para(lx, ly, lz, laminar=True), g, L0, pos, vel=v)
        ch.run_particles(6)
        ref.step(6, istep0=0, nave=3)
        got = ch.particles_get()
        assert np.array_equal(ch.particles_solid(), ref.solid)
        assert np.array_equal(bits(got["pos"].reshape(-1)), bits(ref.X))
        assert np.array_equal(bits(got["vel"].reshape(-1)), bits(ref.V))
        fluid = np.flatnonzero(ref.solid < 0)
        assert np.array_equal(bits(ch.download_post()[:, fluid]), bits(ref.post.reshape(19, -1)[:, fluid]))
