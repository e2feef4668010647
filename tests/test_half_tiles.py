"""Which tiles the workgroups of a launch take whose last round runs as tiles of half the rows (csrc/gemm_tiles.h): the order's own text, compiled for the
host and walked through for every workgroup (tests/half_tiles_check.cpp says what is checked)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "fllm_amd", "csrc")


def test_every_output_is_made_once(tmp_path):
    compiler = shutil.which("g++") or shutil.which("clang++")
    if compiler is None:
        pytest.skip("no host C++ compiler")
    with open(os.path.join(CSRC, "gemm_tiles.h")) as fh:
        place = re.search(r"^template <int EPI, bool GROUPED, int BM, bool HALVES = false>\nstruct Place \{.*?^\};$", fh.read(), re.S | re.M).group(0)
    (tmp_path / "place_host.h").write_text(place)
    binary = str(tmp_path / "half_tiles_check")
    build = subprocess.run([compiler, "-std=c++17", "-O1", "-fsanitize=undefined,address", "-fno-sanitize-recover=all", "-I", str(tmp_path), "-I", CSRC,
                            os.path.join(ROOT, "tests", "half_tiles_check.cpp"), "-o", binary], capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr
    run = subprocess.run([binary], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout + run.stderr
    assert "half tiles ok" in run.stdout
