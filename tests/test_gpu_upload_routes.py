"""GPU test of whole arrays on their way to the device on both sides of the sizes
at which they change their route: up to 2 MiB and from 26 MiB on through the
library's pinned slots (three threads' worth up to 96 MiB), between them by the
runtime's copies, which are faster there; every value arrives."""
import pytest

from shimmed import run_shimmed

pytestmark = pytest.mark.gpu

BODY = """
def slots():
    return ctypes.c_int.in_dll(shim, "shim_host_mallocs").value


MB = 1 << 20
# samples of 44 bytes; slots a trainer of its own allocates
for n, want in ((1489, 0), (1490, 2), (47662, 2), (47663, 0), (300000, 0), (619613, 0), (619614, 6), (700001, 6),
                (2287802, 6), (2287803, 12)):
    assert (want == 0) == (44 * n < 64 << 10 or 2 * MB <= 44 * n < 26 * MB)
    rng = np.random.default_rng(n)
    x, y = rng.random((n, 10), dtype=np.float32), rng.random(n, dtype=np.float32)
    with d3q19.Trainer(n, d3q19.closure_params(1)) as tr:
        before = slots()
        tr.add_samples(x, y)
        assert slots() - before == want, (n, slots() - before)
        fx, fy = tr.samples()
        assert np.array_equal(fx, x) and np.array_equal(fy, y), n
# four fields, rho replaced by the lattice's: below 2 MiB, between, above 26 MiB
for lx, ly, lz in ((32, 32, 63), (32, 32, 65), (77, 101, 45), (64, 128, 103), (64, 128, 105)):
    rng = np.random.default_rng(lz)
    u = [0.01 * rng.standard_normal((lz, ly, lx)) for _ in range(3)]
    with d3q19.Channel(lx, ly, lz) as a, d3q19.Channel(lx, ly, lz) as b:
        for ch in (a, b):
            ch.FORCING()
        a.set_macros(rho=u[0], ux=u[0], uy=u[1], uz=u[2])
        for k, name in enumerate(("ux", "uy", "uz")):
            b.set_macros(**{name: u[k]})
        for ch in (a, b):
            ch.initpop()
            ch.macrovar()
        fa, fb = a.macrovar(download=True), b.macrovar(download=True)
        assert all(np.array_equal(p, q) for p, q in zip(fa, fb))
        half = 0.5 * a.p["force_in_y"] * a.p["force_mag"]
        assert np.max(np.abs(fa[2][:, :, 2:-2].mean() - u[1][:, :, 2:-2].mean() - half)) < 1e-3
"""


def test_routes_and_values(tmp_path):
    run_shimmed(BODY, tmp_path)
