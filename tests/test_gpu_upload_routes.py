"""GPU test of whole arrays on their way to the device on both sides of the sizes
at which they change their route: fields below 2 MiB and from 26 MiB on go
through the library's pinned slots (two for one thread, six for three up to 96
MiB, twelve beyond), between them by the runtime's copies, which are faster
there, and a trainer's samples always by the runtime.  Every value arrives: the
plane sums and the vorticity equal those of a handle whose array was pinned."""
import pytest

from shimmed import run_shimmed

pytestmark = pytest.mark.gpu

BODY = """
hip = ctypes.CDLL("libamdhip64.so.7")
V = ctypes.c_void_p


def slots():
    return ctypes.c_int.in_dll(shim, "shim_host_mallocs").value


for (lx, ly, lz), want in (((16, 16, 31), 0), ((16, 16, 33), 2), ((64, 64, 63), 2), ((64, 64, 65), 0),
                           ((128, 160, 165), 0), ((128, 160, 167), 6), ((256, 256, 191), 6), ((256, 256, 193), 12)):
    N = lx * ly * lz
    rng = np.random.default_rng(lz)
    u = rng.standard_normal((lz, ly, lx))
    p = V()
    assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(8 * N), 0) == 0
    ctypes.memmove(p, u.ctypes.data_as(V), 8 * N)
    got = []
    for pinned in (False, True):
        with d3q19.Channel(lx, ly, lz, "fp16") as ch:
            before = slots()
            assert lib.lbm_set_macros(ch._h, None, p if pinned else u.ctypes.data_as(V), None, None) == 0
            assert slots() - before == (0 if pinned else want), (lx, ly, lz, slots() - before)
            got.append([ch.statistc2()] + (list(ch.vortcalc()) if N < 300000 else []))
    assert np.isfinite(got[0][0]).all() and np.ptp(got[0][0]) > 0
    for a, b in zip(*got):
        assert np.array_equal(a, b), (lx, ly, lz)
    assert hip.hipHostFree(p) == 0

for n in (1, 1490, 50000, 700001):
    rng = np.random.default_rng(n)
    x, y = rng.random((n, 10), dtype=np.float32), rng.random(n, dtype=np.float32)
    with d3q19.Trainer(n, d3q19.closure_params(1)) as tr:
        before = slots()
        tr.add_samples(x, y)
        assert slots() == before, n
        fx, fy = tr.samples()
        assert slots() - before <= 8
        assert np.array_equal(fx, x) and np.array_equal(fy, y), n
"""


def test_routes_and_values(tmp_path):
    run_shimmed(BODY, tmp_path)
