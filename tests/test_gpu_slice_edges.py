"""GPU test of whole populations to and from the host at the edges of the copies'
slices.  A downloaded slice is 1, 2 or 4 MiB (6 656, 13 568 or 27 392 nodes of
152 bytes) for totals below 16 MiB (110 377 nodes), below 64 MiB (441 506) and
from there on, an uploaded one always 4 MiB: exact multiples, one node more, and
totals on both sides of the two changes."""
import numpy as np
import pytest

import d3q19

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lx,ly,lz", [
    (16, 16, 26), (3, 7, 317), (13, 32, 32), (40, 48, 52), (7, 17, 839),      # k x 6 656, one more
    (21, 72, 73), (5, 25, 883), (2, 229, 241),                                # 16 MiB less a few bytes, more
    (48, 48, 53), (39, 49, 71), (53, 64, 80), (47, 73, 87),                   # k x 13 568, one more
    (72, 73, 84), (3, 187, 787),                                              # 64 MiB less, more
    (64, 68, 107), (7, 61, 1283),                                             # k x 27 392, one more
])
def test_round_trips(lx, ly, lz):
    f = 0.01 * np.random.default_rng(lx * ly).standard_normal((lz, ly, lx, 19))
    with d3q19.Channel(lx, ly, lz) as ch:
        ch.upload_f(f)
        assert np.array_equal(ch.download_f(), f)
