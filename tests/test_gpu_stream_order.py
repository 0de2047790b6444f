"""GPU test of the order in which the last handle's streams go: its own after the
host copies' second one, whose queue the runtime would otherwise hand to the
next handle, without the buffers of its own copies."""
import pytest

from shimmed import run_shimmed

pytestmark = pytest.mark.gpu

BODY = """
def get(name):
    return ctypes.c_int.in_dll(shim, name).value


rng = np.random.default_rng(2)
x, y = rng.random((420000, 10), dtype=np.float32), rng.random(420000, dtype=np.float32)
for life in range(4):
    first = get("shim_streams")
    if life % 2 == 0:
        with start(64, 128, 80) as ch:
            ch.macrovar()
            ch.run(2)
            fields, f = ch.macrovar(download=True), ch.download_f()  # 21 and 100 MB
            assert np.max(np.abs(fields[0] - f.sum(-1))) < 1e-15 * 19
    else:
        with d3q19.Trainer(len(y), d3q19.closure_params(1)) as tr:
            tr.add_samples(x, y)
            fx, fy = tr.samples()  # 18.5 MB
            assert np.array_equal(fx, x) and np.array_equal(fy, y)
    assert get("shim_streams") - first == (2 if life % 2 == 0 else 1)
    assert get("shim_last_gone") == first, "the handle's own stream did not go last"
"""


def test_own_stream_goes_last(tmp_path):
    run_shimmed(BODY, tmp_path)
