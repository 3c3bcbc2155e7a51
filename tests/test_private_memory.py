"""The int8 kernels with two positions per workgroup keep what they hold in registers and LDS: the compiler's own report of private memory (spills, arrays
chosen from by a value that is not a constant) says none."""
import os
import re
import subprocess

import pytest

from brokefish_amd import _build


@pytest.mark.parametrize("unit", ["wide512", "ragged256"])
def test_no_private_memory(unit, tmp_path):
    r = subprocess.run([_build.hipcc_path(), *_build.HIPCC_FLAGS, "-Rpass-analysis=kernel-resource-usage", "-I", _build.INCLUDE, "-I", _build.CSRC, "-c",
                        os.path.join(_build.CSRC, f"bf_variant_{unit}.hip"), "-o", str(tmp_path / "unit.o")], check=True, capture_output=True, text=True)
    sizes = re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", r.stderr)
    assert sizes and set(sizes) == {"0"}, r.stderr
