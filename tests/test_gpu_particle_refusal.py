"""GPU test of a particle step that the collision refuses, under a force that
macrovar has not seen: the refused call moves no particle and leaves links,
flags and refilled nodes whole."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads

pytestmark = pytest.mark.gpu


def _start(prec):
    ch = d3q19.Channel(28, 20, 18, prec, laminar=True)
    ux, uy, uz = workloads.laminar_parabola_noise(28, 20, 18, seed=3)
    ch.set_macros(ux=ux, uy=uy, uz=uz)
    ch.FORCING()
    ch.initpop()
    ch.macrovar()
    ch.particles_create(np.array([[8.0, 0.5, 17.5], [8.4, 9.6, 17.0], [20.0, 18.0, 2.0]]),
                        vel=np.array([[0.0, 0.4, 0.0]] * 3), rad=4.6, visc=0.1, nave=4)
    return ch


def _state(ch):
    out = ch.particles_get()
    out["solid"] = ch.particles_solid()
    cap, out["counts"], node, dirs, q = ch.particles_links()
    valid = (np.arange(cap)[None, :] < out["counts"][:, None]).ravel()
    out["node"], out["dirs"], out["q"] = node[valid], dirs[valid], q[valid]
    out["post"] = ch.download_post()
    out["fields"] = np.stack(ch.macrovar(download=True))
    return out


def _same(a, b):
    for k in b:
        assert np.array_equal(a[k], b[k], equal_nan=True), k


@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16"])
def test_force_that_macrovar_has_not_seen(prec):
    with _start(prec) as a, _start(prec) as b:
        for ch in (a, b):
            ch.run_particles(2)
            ch.set_force(0.0, 2.0 * ch.p["force_in_y"], 0.0)
        for _ in range(2):
            with pytest.raises(d3q19.LbmError, match="uniform force that macrovar has seen"):
                a.run_particles(1, istep0=2)
        for ch in (a, b):
            ch.macrovar()
            ch.run_particles(3, istep0=2)
        _same(_state(a), _state(b))
