"""GPU test of the copies to and from arrays that the HIP runtime knows, pinned
by the caller or in device memory: the values are those of ordinary arrays,
and the runtime moves them itself, without the library's pinned slots (but for
several small pinned arrays, whose values alone are checked)."""
import pytest

from shimmed import run_shimmed

pytestmark = pytest.mark.gpu

BODY = """
hip = ctypes.CDLL("libamdhip64.so.7")
V, kind = ctypes.c_void_p, {kind!r}


class Array:
    def __init__(self, values):
        self.a = np.ascontiguousarray(values)
        self.p, n = V(), ctypes.c_size_t(self.a.nbytes)
        # the allocator of the runtime itself: the shim counts the library's calls
        assert (hip.hipMalloc(ctypes.byref(self.p), n) if kind == "device" else
                hip.hipHostMalloc(ctypes.byref(self.p), n, 0)) == 0
        assert hip.hipMemcpy(self.p, self.a.ctypes.data_as(V), n, 1 if kind == "device" else 0) == 0

    def get(self):
        out = np.empty_like(self.a)
        assert hip.hipMemcpy(out.ctypes.data_as(V), self.p, ctypes.c_size_t(out.nbytes),
                             2 if kind == "device" else 0) == 0
        return out


def slots():
    return ctypes.c_int.in_dll(shim, "shim_host_mallocs").value


def ok(rc):
    assert rc == 0, lib.lbm_last_error()


lx, ly, lz = 65, 48, 37  # 3.7 MB of fields
N = lx * ly * lz
pos = np.array([[9.0, 7.0, 8.0], [20.0, 30.0, 25.0]])
for prec in ("fp64", "fp32"):
    post = []
    for plain in (False, True):  # the known arrays first: ordinary ones bring the slots
        with d3q19.Channel(lx, ly, lz, prec) as ch:
            before = slots()
            ch.initpop()
            ch.FORCINGP(7)
            ch.macrovar()
            ch.run(9)
            ch.FORCING()
            ch.macrovar()
            if plain:
                assert np.array_equal(np.stack(ch.macrovar(download=True)), fields)
                assert np.array_equal(ch.download_f(), f) and np.array_equal(ch.download_post(), post)
                ch.set_macros(*fields)
                ch.upload_f(2.0 * f)
                assert np.array_equal(np.stack(ch.macrovar(download=True)), fields2)
                ch.particles_create(pos, rad=4.0)
                assert np.array_equal(ch.particles_solid(), solid)
                assert slots() > before
                continue
            four = [Array(np.zeros(N)) for _ in range(4)]
            ok(lib.lbm_macrovar(ch._h, *[x.p for x in four]))
            assert slots() == before, "the library's slots were used"
            fields = np.stack([x.get().reshape(lz, ly, lx) for x in four])
            fa = Array(np.zeros((lz, ly, lx, 19)))
            ok(lib.lbm_download_f(ch._h, fa.p))
            f = fa.get()
            post = np.empty((19, N))
            if kind == "device" and prec != "fp64":  # widened on the host
                post = ch.download_post()
                before = slots()
            else:
                pa = Array(post)
                ok(lib.lbm_download_post(ch._h, pa.p))
                post = pa.get()
            ok(lib.lbm_set_macros(ch._h, *[x.p for x in four]))
            ok(lib.lbm_upload_f(ch._h, Array(2.0 * f).p))
            ok(lib.lbm_macrovar(ch._h, *[x.p for x in four]))
            fields2 = np.stack([x.get().reshape(lz, ly, lx) for x in four])
            ch.particles_create(pos, rad=4.0)
            sa = Array(np.zeros(N, dtype=np.int32))
            ok(lib.lbm_particles_solid(ch._h, sa.p))
            solid = sa.get()
            assert slots() == before, "the library's slots were used"

rng = np.random.default_rng(3)
x, y = rng.standard_normal((40000, 10)).astype(np.float32), rng.random(40000).astype(np.float32)
with d3q19.Trainer(50000, d3q19.closure_params(1)) as a, d3q19.Trainer(50000, d3q19.closure_params(1)) as b:
    before = slots()
    xa, ya, out, n = Array(x), Array(y), Array(np.zeros(40000, dtype=np.float32)), ctypes.c_longlong()
    ok(lib.lbm_trainer_add_samples(a._h, xa.p, ya.p, 40000))
    ok(lib.lbm_trainer_predict(a._h, 0, 40000, out.p))
    xb, yb = Array(np.zeros_like(x)), Array(np.zeros_like(y))
    ok(lib.lbm_trainer_samples(a._h, ctypes.byref(n), xb.p, yb.p))
    assert slots() == before, "the library's slots were used"
    b.add_samples(x, y)
    assert np.array_equal(out.get(), b.predict(0, 40000))
    assert np.array_equal(xb.get(), x) and np.array_equal(yb.get(), y)
"""


SMALL = BODY.split("lx, ly, lz =")[0] + """
for lx, ly, lz in ((33, 20, 18), (33, 40, 37)):  # 0.4 and 1.6 MB of fields
    with start(lx, ly, lz) as ch:
        ch.macrovar()
        ch.run(3)
        four = [Array(np.zeros((lz, ly, lx))) for _ in range(4)]
        ok(lib.lbm_macrovar(ch._h, *[x.p for x in four]))
        assert np.array_equal(np.stack([x.get() for x in four]), np.stack(ch.macrovar(download=True)))
"""


@pytest.mark.parametrize("kind", ["pinned", "device"])
def test_arrays_the_runtime_knows(kind, tmp_path):
    run_shimmed(BODY.format(kind=kind), tmp_path)


@pytest.mark.parametrize("kind", ["pinned", "device"])
def test_small_fields(kind, tmp_path):
    run_shimmed(SMALL.format(kind=kind), tmp_path)
