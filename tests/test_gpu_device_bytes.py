"""GPU test of lbm_device_bytes against what the library asked the runtime for:
lattices, scratch, fields, and the ring of the blocked sweep."""
import pytest

from shimmed import run_shimmed

pytestmark = pytest.mark.gpu

BODY = """
import os


def asked():
    return ctypes.c_ulonglong.in_dll(shim, "shim_malloc_bytes").value


os.environ["LBM_BLOCK_PLANES"] = "4"
for prec in ("fp64", "fp32", "fp16"):
    for lx, ly, lz in ((2, 1, 1), (12, 10, 6), (33, 20, 18)):
        before = asked()
        with d3q19.Channel(lx, ly, lz, prec) as ch:
            assert ch.device_bytes() == asked() - before, "lattices and scratch"
            ch.FORCING()
            ch.initpop()
            assert ch.device_bytes() == asked() - before, "fields"
            ch.macrovar()
            ch.run(4)
            assert ch.device_bytes() == asked() - before, "the sweep's ring"
"""


def test_every_byte_is_counted(tmp_path):
    run_shimmed(BODY, tmp_path)
