"""GPU test of downloads of a range of the stored lattice: any first node and
length, on and off the 16-byte words and slices that the copies move, against
the whole download; and without the runtime's copies, which odd first nodes
once needed for each population."""
import numpy as np
import pytest

import d3q19
from d3q19 import workloads
from shimmed import run_shimmed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp16", "fp16c"])
@pytest.mark.parametrize("lx,ly,lz", [(7, 5, 3), (33, 65, 31), (101, 93, 61), (130, 131, 129)])
def test_ranges_of_the_lattice(prec, lx, ly, lz):
    N = lx * ly * lz
    rng = np.random.default_rng(N)
    with d3q19.Channel(lx, ly, lz, prec) as ch:
        ch.FORCING()
        ch.upload_f(0.01 * rng.standard_normal((lz, ly, lx, 19)))
        ch.macrovar()
        ch.run(1)
        post = ch.download_post()
        ranges = [(0, N), (0, 1), (N - 1, 1), (1, N - 1), (3, min(N - 3, 50000))]
        ranges += [(int(a), 1 + int(rng.integers(0, min(N - a, 40000)))) for a in rng.integers(0, N, 12)]
        # one population of 64 KiB / 19 and up shares a slot, above 55 188 nodes it has several threads
        ranges += [(f, c) for f in (5, 16) for c in (500, 3457, 55187, 55188, 524288, 1048577) if f + c <= N]
        for first, count in ranges:
            assert np.array_equal(ch.download_post_range(first, count), post[:, first:first + count]), (first, count)


BODY = """
with start(33, 65, 31) as ch:
    ch.macrovar()
    ch.run(1)
    ch.download_post()
    for first in range(17):
        before = ctypes.c_int.in_dll(shim, "shim_copies").value
        ch.download_post_range(22165 + first, 13300)
        assert ctypes.c_int.in_dll(shim, "shim_copies").value == before, first
"""


def test_odd_ranges_use_no_runtime_copies(tmp_path):
    run_shimmed(BODY, tmp_path)
