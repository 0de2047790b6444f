"""GPU tests of kernels that store into pinned slots of the host copies: the
fields at the limits of the slices (64 KiB, 8, 16 and 64 MiB, remainders)
against the oracle's arithmetic on the downloaded populations and against
single fields, whose slices hold other nodes; copies from device addresses
that are not on 16 bytes; values computed node by node through device slices."""
import ctypes

import numpy as np
import pytest

import d3q19

pytestmark = pytest.mark.gpu

CX = np.array([0, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, 1, -1, 1, -1, 0, 0, 0, 0])
CY = np.array([0, 0, 0, 1, -1, 0, 0, 1, 1, -1, -1, 0, 0, 0, 0, 1, -1, 1, -1])
CZ = np.array([0, 0, 0, 0, 0, 1, -1, 0, 0, 0, 0, 1, 1, -1, -1, 1, 1, -1, -1])


# nodes: 2, 2 023, 2 048 (64 KiB of fields), 20 001, 262 144 (8 MiB), 524 288
# (16 MiB), 540 001, 2 097 152 (64 MiB), 2 146 689
@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16c"])
@pytest.mark.parametrize("lx,ly,lz", [(2, 1, 1), (7, 17, 17), (8, 16, 16), (59, 113, 3), (64, 64, 64), (64, 128, 64),
                                      (71, 65, 117), (128, 128, 128), (129, 129, 129)])
def test_fields_in_slices(prec, lx, ly, lz):
    rng = np.random.default_rng(lx * ly + lz)
    shape = (lz, ly, lx)
    with d3q19.Channel(lx, ly, lz, prec) as ch:
        ch.FORCING()
        fy = ch.p["force_in_y"] * ch.p["force_mag"]
        ch.upload_f(0.01 * rng.standard_normal((*shape, 19)))
        f = ch.download_f()  # exactly the stored values
        fields = ch.macrovar(download=True, out=[np.full(shape, np.nan) for _ in range(4)])
        for k in range(4):  # one field alone: four times the nodes in a slice
            one = np.full(shape, np.nan)
            args = [one.ctypes.data_as(ctypes.c_void_p) if j == k else None for j in range(4)]
            d3q19._call("lbm_macrovar", ch._h, *args)
            assert np.array_equal(one, fields[k])
    want = [f.sum(-1), f @ CX, f @ CY + 0.5 * fy, f @ CZ]
    # 19 values below 0.06, added in double or float
    tol = 19 * 19 * 0.06 * (2.0 ** -53 if prec == "fp64" else 2.0 ** -24)
    for a, b in zip(fields, want):
        assert np.max(np.abs(a - b)) <= tol


@pytest.mark.parametrize("pieces", [(1, 7, 4098, 50001), (60000, 3, 60001)])
def test_samples_at_odd_offsets(pieces):
    """40-byte samples: the second and later pieces start off 16 bytes."""
    n = sum(pieces)
    rng = np.random.default_rng(n)
    x, y = rng.standard_normal((n, 10), dtype=np.float32), rng.standard_normal(n, dtype=np.float32)
    with d3q19.Trainer(n, np.zeros(1453, dtype=np.float32)) as t:
        at = 0
        for p in pieces:
            t.add_samples(x[at:at + p], y[at:at + p])
            at += p
        fx, fy = t.samples()
    assert np.array_equal(fx, x) and np.array_equal(fy, y)


def test_closure_inputs_and_viscosity_in_slices():
    """A network of the wall distance alone, whose value changes by 0.02 from
    node to node of a row; 61 does not divide a slice's nodes."""
    lx, ly, lz = 61, 70, 90  # 384 300 nodes: 15.4 MB of inputs, 1.5 MB of viscosities
    rng = np.random.default_rng(8)
    p = np.zeros(1453)
    p[9:320:10], p[352:1376:33], p[1408:1440] = 0.3, 0.25, 0.5
    p[1441:1450], p[1450], p[1451] = 1.0, 100.0, 0.0018
    with d3q19.Channel(lx, ly, lz, "fp32", mrttype=3, visc=0.0018, rstar=60.0) as ch:
        ch.FORCING()
        ch.upload_f(1e-3 * rng.standard_normal((lz, ly, lx, 19)))
        ch.macrovar()
        ch.closure_set(p.astype(np.float32))
        x, nut = ch.closure_inputs()[..., 9].astype(np.float64), ch.closure_nut()
        ystar = ch.p["ystar"]
    wall = np.minimum(np.arange(lx) + 0.5, lx - np.arange(lx) - 0.5) / ystar / 100.0
    assert np.max(np.abs(x - wall)) <= 4 * 2.0 ** -24 * wall.max()
    want = np.logaddexp(0.0, 16.0 * np.tanh(0.25 * np.tanh(0.3 * wall)))
    # half-precision layers: 16 * (0.25 * (2 * 0.54 + 0.5) + 0.13) * 2^-11 below 2^-7
    assert np.max(np.abs(nut - want)) <= 2.0 ** -7
