"""The device headers on the CPU, compiled for the host against a stand-in for
the HIP header (host_stub).

em_device.h: the forms for operands in the middle of the exponent range are
compared bit for bit with the general expressions over random operands and
over flat stencils with an outlier of every size.  em_hostio.h: the transfers
between host arrays and device planes, in pieces and with failing copies.
"""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "emergence_amd", "csrc")


@pytest.mark.parametrize("source", ["device_math_check.cpp", "host_io_check.cpp"])
def test_device_headers_on_the_host(source, tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-w", "-ffp-contract=off", "-I", os.path.join(HERE, "host_stub"), "-I", CSRC,
                    os.path.join(HERE, source), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:]
