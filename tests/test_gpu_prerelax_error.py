"""GPU test of the pre-relaxation loop when a runtime call fails while several
iterations are in flight: what *done and the maxima say is what the lattices
hold, and the handle goes on from there."""
import pytest

from shimmed import run_shimmed

pytestmark = pytest.mark.gpu

BODY = """
lx, ly, lz, n = 97, 97, 97, 10
with start(lx, ly, lz) as b:
    b.rhoupdat()
    b.collision_MRT()
    want = []
    for _ in range(n):
        want.append(b.rhoupdat())
        b.collision_MRT()
eps = want[{last}] if {last} >= 0 else -1.0
with start(lx, ly, lz) as a, start(lx, ly, lz) as b:
    a.rhoupdat()
    a.collision_MRT()
    errs, done = np.full(n, -1.0), ctypes.c_int(-1)
    # two launches an iteration: the first iteration has ended, more are in flight
    switch("shim_fail_query_from", ctypes.c_int.in_dll(shim, "shim_launches").value + 2 * 4)
    switch("shim_fail_query", 1)
    rc = lib.lbm_prerelax(a._h, eps, n, ctypes.byref(done), errs.ctypes.data_as(ctypes.c_void_p))
    assert ctypes.c_int.in_dll(shim, "shim_fail_query").value == 0, "the stream was not asked"
    assert rc != 0 and b"prerelax" in lib.lbm_last_error(), (rc, lib.lbm_last_error())
    k = done.value
    assert 2 <= k < n and (k == {last} + 1 or {last} < 0), k
    assert errs[:k].tolist() == want[:k] and (errs[k:] == -1.0).all(), errs
    b.rhoupdat()
    b.collision_MRT()
    for _ in range(k):
        b.rhoupdat()
        b.collision_MRT()
    assert np.array_equal(bits(a.download_f()), bits(b.download_f()))
    assert a.prerelax(-1.0, 5) == b.prerelax(-1.0, 5)
    a.macrovar()
    b.macrovar()
    a.run(3)
    b.run(3)
    assert np.array_equal(bits(a.download_f()), bits(b.download_f()))
"""


@pytest.mark.parametrize("last", [-1, 1])  # no end among the iterations in flight; the second one ends the loop
def test_state_after_an_error(last, tmp_path):
    run_shimmed(BODY.format(last=last), tmp_path)
