"""GPU test of the lattice size from which pairs of steps run as blocked sweeps
(272 MB, and chunks of at least 88 MB): the report on both sides of it, and
steps, per-call steps and FORCINGP steps there against single steps, bit for
bit in FP64."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads

pytestmark = pytest.mark.gpu


def _state(ch):
    ch.FORCING()
    u = workloads.laminar_parabola_noise(ch.lx, ch.ly, ch.lz, seed=9)
    ch.set_macros(ux=u[0], uy=u[1], uz=u[2])
    ch.initpop()
    ch.macrovar()
    ch.run(5)
    for _ in range(3):
        ch.collision_MRT()
        ch.macrovar()
    ch.run_forcingp(20, 5, 23)
    return ch.download_post()


@pytest.mark.parametrize("prec,lx,ly,lz,pairs", [
    ("fp64", 96, 384, 48, False), ("fp64", 96, 384, 49, True),      # 269 and 275 MB
    ("fp64", 97, 300, 61, False), ("fp64", 97, 300, 62, True),      # 270 and 274 MB, rows off cache lines
    ("fp32", 200, 200, 89, False), ("fp32", 200, 200, 90, True),    # 271 and 274 MB
    ("fp32", 94, 384, 110, False), ("fp32", 95, 384, 110, True),    # chunks of 87.8 and 88.7 MB
    ("fp64", 47, 384, 110, False), ("fp64", 48, 384, 110, True),    # 87.8 and 89.7 MB
])
def test_where_sweeps_begin(monkeypatch, prec, lx, ly, lz, pairs):
    for k in ("LBM_BLOCK_PLANES", "LBM_BLOCK_AXIS", "LBM_BLOCK_ROWS", "LBM_BLOCK_FORCED", "LBM_DEFER"):
        monkeypatch.delenv(k, raising=False)
    with d3q19.Channel(lx, ly, lz, prec) as a:
        assert a.block_pairs() == pairs
        if not pairs:
            return
        before = a.device_bytes()
        pa = _state(a)
        assert a.device_bytes() > before, "no pair has run"
    monkeypatch.setenv("LBM_BLOCK_PLANES", "0")
    with d3q19.Channel(lx, ly, lz, prec) as b:
        assert not b.block_pairs()
        pb = _state(b)
    if prec == "fp64":
        assert np.array_equal(pa, pb)
    else:  # FMA contraction may differ between the kernels: an ulp of the largest value a step
        assert np.max(np.abs(pa - pb)) <= 13 * 2.0 ** -23 * np.max(np.abs(pb))
