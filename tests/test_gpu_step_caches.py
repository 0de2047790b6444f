"""GPU test of single steps at the sizes where their loads and stores take
another way through the caches.  A flow that repeats along z stays so: every
period of the tall channel equals the channel of one period, whose lattice is
small enough for the plainest of the ways."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads

pytestmark = pytest.mark.gpu

LX, LY, LZ = 97, 97, 8


def _flow(prec, periods):
    u = workloads.laminar_parabola_noise(LX, LY, LZ, seed=12)
    v = [0.5 * a for a in u]
    tall = [[np.concatenate([a] * periods, axis=0) for a in w] for w in (u, v)]
    with d3q19.Channel(LX, LY, LZ * periods, prec) as ch:
        ch.FORCING()
        ch.set_macros(ux=tall[0][0], uy=tall[0][1], uz=tall[0][2])
        ch.initpop()
        ch.macrovar()
        ch.run(5)
        for _ in range(3):
            ch.collision_MRT()
            ch.macrovar()
        ch.set_macros(ux=tall[1][0], uy=tall[1][1], uz=tall[1][2])
        ch.collision_MRT()  # a step with stored fields
        ch.collision_MRT()
        return ch.download_f()


# one lattice of 75 k nodes: 11 MB in FP64, 6 MB in FP32; tall ones with both
# lattices in the L2s, both in the last-level cache, one in it, and larger
@pytest.mark.parametrize("prec,periods", [("fp64", 2), ("fp64", 11), ("fp64", 12), ("fp64", 24), ("fp64", 27),
                                          ("fp32", 2), ("fp32", 3), ("fp32", 22), ("fp32", 25), ("fp32", 53)])
def test_tall_channel_equals_its_period(prec, periods):
    one, tall = _flow(prec, 1), _flow(prec, periods)
    f = tall.reshape((periods,) + one.shape)
    if prec == "fp64":
        assert np.array_equal(np.ascontiguousarray(f).view(np.uint64),
                              np.ascontiguousarray(np.broadcast_to(one, f.shape)).view(np.uint64))
    else:  # FMA contraction may differ between the kernels: an ulp of the largest value
        assert np.max(np.abs(f - one)) <= 1e-6 * np.max(np.abs(one))
