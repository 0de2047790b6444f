"""The per-call main loop where its pairs really run as blocked sweeps: small
lattices take single steps unless the sweep's variables ask for it, so these
handles set LBM_BLOCK_PLANES.  Every interleaving of calls leaves the state of
a handle that launches each collision at once (LBM_DEFER=0), bit for bit, and
the plain loop that of the oracle.  That a pair has run shows in the ring that
the first one allocates."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads
import oracle as O
from test_gpu_percall import OPS, _apply, bits

pytestmark = pytest.mark.gpu


def _channel(monkeypatch, lx, ly, lz, prec="fp64", defer="1", axis=None):
    monkeypatch.setenv("LBM_BLOCK_PLANES", "4")
    monkeypatch.setenv("LBM_DEFER", defer)
    if axis:
        monkeypatch.setenv("LBM_BLOCK_AXIS", axis)
    ch = d3q19.Channel(lx, ly, lz, prec)
    for k in ("LBM_BLOCK_PLANES", "LBM_DEFER", "LBM_BLOCK_AXIS"):
        monkeypatch.delenv(k, raising=False)
    return ch


def _pair(monkeypatch, lx, ly, lz, prec="fp64", seed=5, axis=None):
    out = [_channel(monkeypatch, lx, ly, lz, prec, d, axis) for d in ("1", "0")]
    vel = workloads.laminar_parabola_noise(lx, ly, lz, seed=seed, uc=0.04)
    for c in out:
        c.set_macros(ux=vel[0], uy=vel[1], uz=vel[2])
        c.FORCING()
        c.initpop()
        c.macrovar()
    return out


def test_pairs_are_reported_as_they_run(monkeypatch):
    for k in ("LBM_BLOCK_PLANES", "LBM_BLOCK_AXIS", "LBM_BLOCK_ROWS", "LBM_DEFER"):
        monkeypatch.delenv(k, raising=False)
    with _channel(monkeypatch, 24, 20, 18) as swept, d3q19.Channel(24, 20, 18) as single, \
            d3q19.Channel(24, 20, 18, "fp16") as none:
        for ch, pairs in ((swept, True), (single, False), (none, False)):
            assert ch.block_pairs() == pairs
            ch.FORCING()
            ch.initpop()
            before = ch.device_bytes()
            ch.macrovar()
            ch.run(2)
            assert (ch.device_bytes() > before) == pairs


@pytest.mark.parametrize("lx,ly,lz", [(32, 64, 32), (19, 14, 11)])
@pytest.mark.parametrize("axis", ["z", "y"])
def test_per_call_loop_equals_the_oracle(monkeypatch, axis, lx, ly, lz):
    ref = O.OracleChannel(lx, ly, lz)
    ref.FORCING()
    ref.ux[:], ref.uy[:], ref.uz[:] = workloads.laminar_parabola_noise(lx, ly, lz, seed=61)
    ref.initpop()
    f0 = ref.f.copy()
    ref.macrovar()
    for _ in range(41):
        ref.collision_MRT()
        ref.macrovar()
    with _channel(monkeypatch, lx, ly, lz, axis=axis) as ch:
        ch.upload_f(f0)
        ch.FORCING()
        ch.macrovar()
        before = ch.device_bytes()
        for _ in range(41):  # 20 pairs and a single step
            ch.collision_MRT()
            ch.macrovar()
        assert ch.device_bytes() > before, "no pair has run"
        assert np.array_equal(bits(ch.download_f()), bits(ref.f))
        for a, b in zip(ch.macrovar(download=True), (ref.rho, ref.ux, ref.uy, ref.uz)):
            assert np.array_equal(bits(a), bits(b))


@pytest.mark.parametrize("seed", [1, 2, 3, 4])
@pytest.mark.parametrize("axis", ["z", "y"])
def test_random_call_sequences_match_undeferred_calls(monkeypatch, axis, seed):
    lx, ly, lz = (24, 20, 18) if seed % 2 else (19, 14, 11)
    rng = np.random.default_rng(seed)
    ops = [OPS[i] for i in rng.integers(0, len(OPS), 120)]
    ops = ["coll", "mac"] * 6 + ops + ["coll", "mac", "coll", "mac", "coll"]
    a, b = _pair(monkeypatch, lx, ly, lz, seed=seed, axis=axis)
    with a, b:
        before = [c.device_bytes() for c in (a, b)]
        for k, op in enumerate(ops):
            ra, rb = _apply(a, op, k), _apply(b, op, k)
            if ra is not None:
                assert np.array_equal(bits(ra), bits(rb)), f"step {k}: {op}"
            if k == 11:  # the six steps: three pairs on a, none on b
                assert a.device_bytes() > before[0] and b.device_bytes() == before[1]
        assert np.array_equal(bits(a.download_f()), bits(b.download_f()))
        assert np.array_equal(bits(a.download_post()), bits(b.download_post()))


@pytest.mark.parametrize("prec", ["fp32", "fp16", "fp16c"])
def test_per_call_loop_reduced_precision(monkeypatch, prec):
    """Pairs, by request in 2-byte storage too, against single steps, whose FMA
    contraction may differ: an ulp of the largest value per step."""
    a, b = _pair(monkeypatch, 24, 20, 18, prec=prec)
    with a, b:
        before = a.device_bytes()
        for c in (a, b):
            for _ in range(9):
                c.collision_MRT()
                c.macrovar()
        assert a.device_bytes() > before, "no pair has run"
        pa, pb = a.download_post(), b.download_post()
    ulp = 2.0 ** -23 if prec == "fp32" else 2.0 ** -10
    assert np.max(np.abs(pa - pb)) <= 9 * ulp * np.max(np.abs(pb))


@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16", "fp16c"])
@pytest.mark.parametrize("axis", ["z", "y"])
def test_forcingp_steps_one_by_one_then_swept(monkeypatch, prec, axis):
    """LBM_BLOCK_FORCED=0: lbm_run_forcingp runs FORCINGP steps one by one and
    the FORCING steps after npforcing in pairs; against the calls one by one,
    in FP32 and 2-byte storage with the tolerance of a contraction that differs."""
    lx, ly, lz = 20, 18, 14
    vel = workloads.laminar_parabola_noise(lx, ly, lz, seed=35)
    out = []
    monkeypatch.setenv("LBM_BLOCK_FORCED", "0")
    a = _channel(monkeypatch, lx, ly, lz, prec, "0", axis)
    monkeypatch.delenv("LBM_BLOCK_FORCED", raising=False)
    b = _channel(monkeypatch, lx, ly, lz, prec, "0", axis)
    with a, b:
        for c in (a, b):
            c.set_macros(ux=vel[0], uy=vel[1], uz=vel[2])
            c.FORCING()
            c.initpop()
            c.macrovar()
        before = a.device_bytes()
        a.run_forcingp(20, 14, 35)
        assert a.device_bytes() == before, "a FORCINGP step was swept"
        b.run_forcingp_stepwise(20, 14, 35)
        assert b.device_bytes() == before
        a.run_forcingp(34, 11, 35)
        assert a.device_bytes() > before, "no FORCING pair has run"
        b.run_forcingp_stepwise(34, 11, 35)
        out = [c.download_post() for c in (a, b)]
        fields = [np.stack(c.macrovar(download=True)) for c in (a, b)]
    if prec == "fp64":
        assert np.array_equal(bits(out[0]), bits(out[1])) and np.array_equal(bits(fields[0]), bits(fields[1]))
    else:
        ulp = 2.0 ** -23 if prec == "fp32" else 2.0 ** -10
        assert np.max(np.abs(out[0] - out[1])) <= 25 * ulp * np.max(np.abs(out[1]))
