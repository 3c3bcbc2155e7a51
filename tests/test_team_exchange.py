"""The exchanges of the team form, on the CPU: a wavefront's flag stands for what that wavefront itself stored, so
every byte a reader loads must have been stored by a wavefront whose flag the reader waited for.  The host program
walks the layout functions the kernel is compiled with, for both network widths."""
import os
import subprocess

from brokefish_amd import _build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_load_of_the_second_exchange_waits_for_its_store(tmp_path):
    exe = str(tmp_path / "team_exchange_check")
    subprocess.run([_build.hipcc_path(), "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-Wno-unused-command-line-argument",
                    "-I", _build.INCLUDE, "-I", _build.CSRC, os.path.join(HERE, "abi", "team_exchange_check.hip"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
    assert "width 256" in run.stdout and "width 512" in run.stdout
