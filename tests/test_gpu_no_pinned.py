"""GPU test of every call whose small result goes through pinned memory, and of
the host copies, when no pinned memory is to be had: the same values."""
import pytest

from shimmed import run_shimmed

pytestmark = pytest.mark.gpu

CHANNEL = """
def values(prec):
    out = {}
    with start(24, 20, 18, prec) as ch:
        out["prerelax"] = ch.prerelax(-1.0, 70)
        out["rhoupdat"] = ch.rhoupdat()
        assert lib.lbm_rhoupdat(ch._h, None) == 0
        ch.collision_MRT()
        ch.macrovar()
        ch.run(5)
        out["mass"], out["ave"], out["diag"] = ch.mass(), ch.avedensity(), ch.diag()
        out["stat"], out["diss"] = ch.statistc2(), ch.dissipation()
        ch.stats_accumulate()
        ch.stats_accumulate_filtered()
        out["run"], out["filtered"] = ch.stats_read()[0], ch.stats_read_filtered()[0]
        ch.macrovar()
        out["fields"], out["f"], out["post"] = np.stack(ch.macrovar(download=True)), ch.download_f(), ch.download_post()
        ch.upload_f(out["f"])
        ch.macrovar()
        ch.particles_create(np.array([[8.0, 6.0, 6.0], [16.0, 14.0, 12.0]]), rad=3.5)
        ch.run_particles(3)
        out.update(ch.particles_get())
        out["solid"] = ch.particles_solid()
    return out


for prec in ("fp64", "fp32"):
    want = values(prec)
    switch("shim_fail_host_malloc", 1)
    got = values(prec)
    switch("shim_fail_host_malloc", 0)
    assert set(got) == set(want)
    for k in want:
        assert np.array_equal(got[k], want[k], equal_nan=True), (prec, k)
"""

TRAINER = """
rng = np.random.default_rng(3)
x, y = rng.standard_normal((40000, 10)).astype(np.float32), rng.random(40000).astype(np.float32)


def values():
    with d3q19.Trainer(50000, d3q19.closure_params(1)) as t:
        t.add_samples(x, y)
        out = [*t.grad(0, 30000), t.train(0, 40000, 3, 4096, 1e-3), t.params(), t.predict(0, 40000)]
        return out + list(t.samples())


want = values()
switch("shim_fail_host_malloc", 1)
got = values()
assert len(got) == len(want) and all(np.array_equal(a, b) for a, b in zip(got, want))
"""


def test_channel_results_without_pinned_memory(tmp_path):
    run_shimmed(CHANNEL, tmp_path)


def test_trainer_results_without_pinned_memory(tmp_path):
    run_shimmed(TRAINER, tmp_path)
