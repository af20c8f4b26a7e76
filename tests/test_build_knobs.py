"""Build-time sizes that the kernels divide evenly: a value that they would
cut short does not compile."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gaussian-point-splatting_amd", "csrc")


@pytest.mark.parametrize("tiles,compiles", [("512u", True), ("1000u", False)])
def test_fold_tiles(tmp_path, tiles, compiles):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is not available")
    src = tmp_path / "knob.hip"
    src.write_text('#include "gps_internal.h"\n')
    r = subprocess.run([hipcc, "-std=c++17", "--offload-arch=gfx950", "-fsyntax-only", "-I", CSRC,
                        "-DGPS_FOLD_TILES=" + tiles, str(src)], capture_output=True, text=True, timeout=120)
    assert (r.returncode == 0) == compiles, r.stderr
    assert compiles or "same number of tiles" in r.stderr
