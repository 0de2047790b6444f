"""GPU test of the host copies' second stream: only copies of 256 MiB and more
make one, and their values are those of smaller copies."""
import pytest

from shimmed import run_shimmed

pytestmark = pytest.mark.gpu

BODY = """
def streams():
    return ctypes.c_int.in_dll(shim, "shim_streams").value


# 0.1, 21, 100 (the populations) and 273 MB of fields
for (lx, ly, lz), made in (((16, 16, 16), 1), ((64, 128, 80), 1), ((16, 16, 16), 1), ((64, 128, 80), 1),
                           ((256, 256, 130), 2)):
    before = streams()
    with start(lx, ly, lz) as ch:
        ch.macrovar()
        ch.run(2)
        fields = ch.macrovar(download=True)
        if lz < 100:
            f = ch.download_f()
            assert np.max(np.abs(fields[0] - f.sum(-1))) < 1e-15 * 19
        one = np.empty((lz, ly, lx))
        for k in range(4):
            args = [one.ctypes.data_as(ctypes.c_void_p) if j == k else None for j in range(4)]
            d3q19._call("lbm_macrovar", ch._h, *args)
            assert np.array_equal(one, fields[k]), k
    assert streams() - before == made, (lx, streams() - before)
"""


def test_streams_of_a_life(tmp_path):
    run_shimmed(BODY, tmp_path)
