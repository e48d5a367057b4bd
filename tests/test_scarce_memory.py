"""The library without device memory, pinned memory or threads to spare
(tests/selftest/tlm_scarce.cpp): the same results by its other routes, no error
left behind, and its usual routes again as soon as there is room. Without a GPU
the program reports SKIP and succeeds."""
import os
import subprocess

import pytest

from emsolver_amd import tlm

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "selftest", "tlm_scarce")


def _run():
    assert os.path.exists(EXE), "build the test programs first (__graft_entry__.build())"
    p = subprocess.run([EXE], capture_output=True, text=True, timeout=100)
    print(p.stdout)
    return p


@pytest.mark.skipif(tlm.device_count() > 0, reason="a HIP device is present")
def test_without_device_skips():
    p = _run()
    assert p.returncode == 0 and "SKIP" in p.stdout


@pytest.mark.gpu
def test_scarce_memory_on_gpu():
    p = _run()
    assert "FAIL" not in p.stdout, p.stdout
    assert p.returncode == 0 and "SCARCETEST PASSED" in p.stdout
