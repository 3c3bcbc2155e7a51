"""The exchanges of the team form, on the CPU: a wavefront's flag stands for what that wavefront itself stored, so
every byte a reader loads must have been stored by a wavefront whose flag the reader waited for.  The host program
walks the layout functions the kernel is compiled with, for both network widths."""
import os
import subprocess

import pytest

from brokefish_amd import _build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def checked(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("team") / "team_exchange_check")
    subprocess.run([_build.hipcc_path(), "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-Wno-unused-command-line-argument",
                    "-I", _build.INCLUDE, "-I", _build.CSRC, os.path.join(HERE, "abi", "team_exchange_check.hip"), "-o", exe], check=True)
    return subprocess.run([exe], capture_output=True, text=True).stdout


def test_every_load_of_the_second_exchange_waits_for_its_store(checked):
    for width in (256, 512):
        assert any(line.startswith(f"width {width}:") and line.endswith(" 0 faults") for line in checked.splitlines()), checked


def test_flags_are_told_from_earlier_ones_where_the_count_wraps(checked):
    assert "counts: 0 faults" in checked, checked


def test_the_form_is_used_only_where_a_process_leaves_units_to_complete_a_team(checked):
    assert "units: 0 faults" in checked, checked
