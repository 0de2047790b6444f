"""GPU test of lbm_particles_get with more particles than the handle's small
buffer holds: it allocates nothing, so no C++ exception can leave the C ABI."""
import pytest

from shimmed import run_shimmed

pytestmark = pytest.mark.gpu

BODY = """
np_ = 120
pos = np.stack([np.tile([6.0, 18.0], 60), np.repeat(6.0 * np.arange(12) + 3.0, 10),
                np.tile(np.repeat(6.0 * np.arange(5) + 3.0, 2), 12)], axis=1)
assert len(pos) == np_ and 24 * np_ > 12 * 24
with start(24, 72, 30) as ch:
    ch.macrovar()
    ch.particles_create(pos, rad=2.0)
    ch.run_particles(2)
    want = ch.particles_get()
    ctypes.c_ulonglong.in_dll(shim, "shim_fail_new").value = (24 * np_ + 1) * 8
    got = ch.particles_get()
    for k in want:
        assert np.array_equal(got[k], want[k]), k
"""


def test_many_particles(tmp_path):
    run_shimmed(BODY, tmp_path)
