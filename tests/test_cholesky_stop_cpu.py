"""The stop of the AO Cholesky decomposition: block 0 raises the stop flag in
the launch that finds nothing above the threshold, while other blocks of that
launch may be starting, so that the waves of one block read either value.
The kernel is built for the host and a block's waves are released before and
after the flag in every combination: the step must leave everything as it was."""
import os
import subprocess

from conftest import ROOT


def test_waves_of_a_block_stop_together(tmp_path):
    exe = tmp_path / "chol_panel_host"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "dalton_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "chol_panel_host.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
