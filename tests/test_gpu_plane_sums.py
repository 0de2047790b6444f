"""GPU test of the plane sums (statistc2, the box-filtered running statistics,
dissipation_calc) and of diag's final sums where their work split changes: one
column tile and several, columns that do not fill a wave, fewer rows than
chunks, row lanes without a row, grids of fewer blocks than diag's partials.

Tolerance: all sums are FP64 over at most ly*lz terms of one sign or of
products of fields; two orders of n additions differ by at most n * 2^-53 of
the sum of magnitudes (n < 3 000: 4e-13), and the columns subtract products of
means of the same size; 1e-11 of a column's largest value covers both."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads
import oracle as O

pytestmark = pytest.mark.gpu


def _close(got, want, what):
    scale = np.abs(want).max(axis=0)
    assert np.all(np.abs(got - want) <= 1e-11 * scale), (what, np.abs(got - want).max(0) / np.maximum(scale, 1e-300))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("lx,ly,lz", [(2, 2, 2), (16, 2, 4), (62, 30, 34), (64, 6, 4), (66, 40, 26), (130, 34, 62),
                                      (192, 12, 10), (254, 8, 6), (258, 10, 8), (300, 46, 52)])
def test_plane_sums_at_split_edges(prec, lx, ly, lz):
    with d3q19.Channel(lx, ly, lz, prec) as ch:
        ux, uy, uz = workloads.laminar_parabola_noise(lx, ly, lz, seed=4, amp=0.3)
        ch.set_macros(ux=ux, uy=uy, uz=uz)
        ch.FORCING()
        ch.initpop()
        ch.macrovar()
        ch.run(3)
        ch.stats_accumulate_filtered()
        got = {"statistc2": ch.statistc2(), "filtered": ch.stats_read_filtered()[0], "dissipation": ch.dissipation()}
        diag = ch.diag()
        rho, *u = ch.macrovar(download=True)
        f = ch.download_f()
        us, ystar = ch.p["ustar"], ch.p["ystar"]

    def profile(rho, u):
        m = lambda a: a.mean(axis=(0, 1))  # noqa: E731
        v = [m(a) / us for a in u]
        c = lambda a, b: m(u[a] * u[b]) / us**2 - v[a] * v[b]  # noqa: E731
        p = m(rho) / us**2
        return np.stack([*v, c(0, 0), c(1, 1), c(2, 2), c(0, 2), c(0, 1), c(1, 2), p,
                         m(rho * rho) / us**4 - p * p], 1)

    # magnitudes of the terms summed (of the fine nodes, for the filtered fields too); the variances are
    # differences of means of squares
    size = np.array([max(np.abs(a).max() for a in u) / us] * 3 + [max((a * a).max() for a in u) / us**2] * 6
                    + [np.abs(rho).max() / us**2, (rho * rho).max() / us**4])

    def against(got, rho, u, what):
        assert np.all(np.abs(got[:, 2:13] - profile(rho, u)) <= 1e-11 * size), what

    box = lambda a: a.reshape(lz // 2, 2, ly // 2, 2, lx // 2, 2).mean(axis=(1, 3, 5))  # noqa: E731
    against(got["statistc2"], rho, u, "statistc2")
    against(got["filtered"], box(rho), [box(a) for a in u], "filtered")
    o = O.OracleChannel(lx, ly, lz)
    o.rho[:], o.ux[:], o.uy[:], o.uz[:], o.f[:] = rho, *u, f
    if prec == "fp64":
        _close(got["dissipation"], o.dissipation(), "dissipation")
        speed = np.sqrt(u[0]**2 + u[1]**2 + u[2]**2)
        assert diag[0] == speed.max() and diag[11] == rho.max() and diag[12] == rho.min()
        means = np.array([a.mean() for a in u]) / us
        assert np.all(np.abs(diag[4:7] - means) <= 1e-12 * max(np.abs(a).max() for a in u) / us)
