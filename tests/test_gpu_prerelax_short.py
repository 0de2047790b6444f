"""GPU test of pre-relaxations that end at their first iteration, as they do from
initpop's populations: no iteration is launched after it, and the state is that
of the two calls."""
import pytest

from shimmed import run_shimmed

pytestmark = pytest.mark.gpu

BODY = """
def launches():
    return ctypes.c_int.in_dll(shim, "shim_launches").value


for prec in ("fp64", "fp32"):
    with start(33, 20, 18, prec) as a, start(33, 20, 18, prec) as b:
        b.rhoupdat()
        before = launches()
        b.collision_MRT()
        assert launches() - before == 1, "launches are not counted"
        before = launches()
        it, err = a.prerelax()
        assert it == 0 and err <= 1e-5
        assert launches() - before == 2, launches() - before  # the iteration and its maximum
        assert np.array_equal(bits(a.download_f()), bits(b.download_f()))
"""


def test_one_iteration_is_one_launched(tmp_path):
    run_shimmed(BODY, tmp_path)
