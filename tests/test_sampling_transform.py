"""The splat's sampling transform against the general deterministic functions
it stands for (tests/sampling_check.cpp, the renderer's own headers compiled
with g++ as the CPU oracle is), bit for bit."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "gaussian-point-splatting_amd", "csrc")


@pytest.fixture(scope="module")
def counts(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ is not available")
    exe = str(tmp_path_factory.mktemp("sampling") / "sampling_check")
    subprocess.run([gxx, "-std=c++17", "-O2", "-march=native", "-ffp-contract=off", "-fno-fast-math", "-I", CSRC, "-o",
                    exe, os.path.join(HERE, "sampling_check.cpp")], check=True)
    return [int(v) for v in subprocess.run([exe, "4000000"], check=True, capture_output=True, text=True).stdout.split()]


@pytest.mark.parametrize("what", ["logs", "angles", "points"])
def test_sampling_transform_same_bits(counts, what):
    assert counts[("logs", "angles", "points").index(what)] == 0
