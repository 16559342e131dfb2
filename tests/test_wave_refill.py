"""The refill rules of the one-lane traversal walk, compiled for the host from
the kernels' own header: every wave of a launch ends and every ray is traced
once, whatever the number of rays, of waves and of rays that are to be traced
again (a wave of a small launch owns fewer lanes than it may park)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "firefly_amd", "csrc")


def test_every_wave_ends(tmp_path):
    exe = str(tmp_path / "wave_refill")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", CSRC, os.path.join(HERE, "wave_refill.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
