"""Contexts on two devices in one process keep their buffers on their own
device, on the CPU with a stand-in for the HIP runtime (tests/fake_hip.hpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "parallel-ra_amd")


@pytest.mark.skipif(not os.path.exists(os.path.join(PKG, "libpra_amd.so")), reason="libpra_amd.so not built")
def test_buffers_lie_on_their_contexts_device(tmp_path):
    exe = str(tmp_path / "two_devices_test")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-O1", "-rdynamic", "-I" + os.path.join(ROOT, "include"),
                    "-o", exe, os.path.join(ROOT, "tests", "two_devices_test.cpp"), "-L" + PKG, "-lpra_amd",
                    "-Wl,-rpath," + PKG, "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
