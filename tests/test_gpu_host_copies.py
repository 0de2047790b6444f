"""GPU tests of the copies between device lattices and host arrays: exact
round trips at sizes around the limits of their slices (below and above 1
MiB, 8 MiB, one and several 4 MiB slices, with remainders), the widening
lattice download against ranges of itself, and two handles copying from two
threads at once (one copy uses the shared pinned buffers, the other goes the
plain way)."""
import threading

import numpy as np
import pytest

import d3q19

pytestmark = pytest.mark.gpu


def _lattice(lx, ly, lz, seed):
    return 0.01 * np.random.default_rng(seed).standard_normal((lz, ly, lx, 19))


# f bytes = 152 N: 0.9, 1.05, 8.3, 8.5 and 41.2 MiB (slices of 27 392 nodes)
@pytest.mark.parametrize("lx,ly,lz", [(16, 25, 15), (16, 27, 17), (33, 42, 42), (107, 32, 16), (32, 107, 16),
                                      (64, 64, 69)])
def test_round_trips_at_slice_edges(lx, ly, lz):
    f = _lattice(lx, ly, lz, lx)
    with d3q19.Channel(lx, ly, lz) as ch:
        ch.upload_f(f)
        assert np.array_equal(ch.download_f(), f)
        ch.macrovar()
        fields = ch.macrovar(download=True)
        ch.set_macros(*[a + 1.0 for a in fields])
        ch.rhoupdat()  # rho from the lattice; u stays what was set
        post = ch.download_post()
        n = lx * ly * lz
        assert np.array_equal(post[:, n // 3:n // 2], ch.download_post_range(n // 3, n // 2 - n // 3))
        vort = ch.vortcalc()
        again = ch.vortcalc()
        assert all(np.array_equal(a, b) for a, b in zip(vort, again))


@pytest.mark.parametrize("prec,bits", [("fp32", 24), ("fp16", 11), ("fp16c", 12)])
def test_widening_download(prec, bits):
    """Stored values come back as the FP64 value of the stored word; 1 100 000
    nodes give several slices a population in FP32, one in 2-byte storage."""
    lx, ly, lz = 100, 110, 100
    f = _lattice(lx, ly, lz, 5)
    with d3q19.Channel(lx, ly, lz, prec) as ch:
        ch.upload_f(f)
        g = ch.download_f()
        assert np.max(np.abs(g - f)) <= np.abs(f).max() * 2.0 ** -bits
        ch.upload_f(g)  # representable now
        post = ch.download_post()
        assert np.array_equal(ch.download_f(), g)
    # rest populations do not move: post[0] is f0 node by node
    assert np.array_equal(post[0], g[..., 0].reshape(-1))


def test_two_threads_copy_at_once():
    shapes = [(48, 64, 50), (52, 60, 56)]
    ok = [False, False]

    def work(k):
        f = _lattice(*shapes[k], 70 + k)
        with d3q19.Channel(*shapes[k]) as ch:
            good = True
            for r in range(6):
                ch.upload_f(f + r)
                good = good and np.array_equal(ch.download_f(), f + r)
                ch.macrovar()
                rho = ch.macrovar(download=True)[0]
                good = good and np.allclose(rho, (f + r).sum(-1), rtol=0, atol=1e-12 * (19 * (r + 1)))
            ok[k] = good

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    assert ok == [True, True]


def test_pool_survives_its_last_user():
    """The pinned buffers go with the last handle and come back with the next."""
    f = _lattice(40, 50, 60, 9)
    for _ in range(3):
        with d3q19.Channel(40, 50, 60) as ch:
            ch.upload_f(f)
            assert np.array_equal(ch.download_f(), f)
