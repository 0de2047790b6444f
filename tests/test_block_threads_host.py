"""Host-side check of the blocked sweep's threads (tests/host/block_threads_check.hip),
compiled with hipcc and run on the CPU; no GPU involved."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"),
                    reason="hipcc not available")
def test_threads_of_the_sweep_with_padded_populations(tmp_path):
    """The kernel's thread mapping, with shifted z slabs and the padded stride of
    the populations: bounds, single writes, step t+2 everywhere, whole lines."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    exe = os.path.join(tmp_path, "block_threads_check")
    subprocess.run([hipcc, "-O2", "-std=c++17", "-I", os.path.join(ROOT, "d3q19-single-phase_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "block_threads_check.hip"), "-o", exe],
                   check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr + r.stdout
    assert "ok sweep threads" in r.stdout
