"""Offsets that leave 32 bits on the largest domains (mom5_amd/csrc/planes.h),
checked on the host."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "mom5_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_plane_offsets(tmp_path):
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", CSRC,
                    os.path.join(ROOT, "tests", "planes_check.cpp"), "-o",
                    str(tmp_path / "planes_check")], check=True)


@pytest.mark.parametrize("source", ["k_quicker.hip", "k_quick_step.hip"])
def test_quicker_weights_have_64_bit_plane_offsets(source):
    """The 16 planes of Quicker weights are written when a context is created and
    read by the Quicker kernels: P2 is an int, and 15 * P2 leaves it from 2^27.2
    points a level on (12000 x 12000), well inside what mom_gpu_create takes."""
    text = open(os.path.join(CSRC, source)).read()
    assert not re.search(r"\bw\[[^]]*\* *P2", text)
    assert not re.search(r"\bqw\[[^]]*\* *P2", text)
