"""The arithmetic of the device headers on the CPU: em_device.h is compiled for
the host against a stand-in for the HIP header (host_stub), and the forms for
operands in the middle of the exponent range are compared bit for bit with the
general expressions over random operands and over flat stencils with an
outlier of every size."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "emergence_amd", "csrc")


def test_mid_range_forms_give_the_general_bits(tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-w", "-ffp-contract=off", "-I", os.path.join(HERE, "host_stub"), "-I", CSRC,
                    os.path.join(HERE, "device_math_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:]
