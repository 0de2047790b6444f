"""GPU test of the FP32 steps with 32-bit offsets (csrc/kernels_impl.h:
pull32): lattices that the last-level cache cannot hold take them, and
LBM_STEP_W32=0 the 64-bit form, which loads and stores the same values, so the
stored words are the same bit for bit.  Odd sizes, so that waves hold lanes at
both walls, and every mode of the step that takes the form."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads

pytestmark = pytest.mark.gpu

GRID = (97, 251, 171)  # 4.2 M nodes, a lattice of 316 MB


@pytest.mark.parametrize("case", ["plain", "rho_offset", "arrays", "forcingp", "particles", "prerelax"])
def test_fp32_forms_store_the_same_words(monkeypatch, case):
    monkeypatch.setenv("LBM_BLOCK_PLANES", "0")  # single steps
    u = workloads.laminar_parabola_noise(*GRID, seed=6)
    posts = []
    for env in (None, "0"):
        if env is None:
            monkeypatch.delenv("LBM_STEP_W32", raising=False)
        else:
            monkeypatch.setenv("LBM_STEP_W32", env)
        with d3q19.Channel(*GRID, "fp32", laminar=True) as ch:
            ch.FORCING()
            ch.set_macros(ux=u[0], uy=u[1], uz=u[2])
            ch.initpop()
            if case == "prerelax":
                ch.prerelax(-1.0, 2)
            elif case == "arrays":
                for _ in range(3):
                    ch.rhoupdat()
                    ch.collision_MRT()
            else:
                ch.macrovar()
                if case == "plain":
                    ch.run(5)
                elif case == "rho_offset":
                    for _ in range(3):
                        ch.avedensity()
                        ch.collision_MRT()
                        ch.macrovar()
                elif case == "forcingp":
                    ch.run_forcingp(0, 4, 10)
                else:
                    ch.particles_create(np.array([[30.0, 0.4, 170.6], [60.2, 125.0, 85.0]]), rad=5.0, nave=2)
                    ch.run_particles(5)
            posts.append(ch.download_post().astype(np.float32))
    assert np.array_equal(posts[0].view(np.uint32), posts[1].view(np.uint32))
