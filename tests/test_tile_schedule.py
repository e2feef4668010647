"""The order of loads, waits, barriers and LDS reads in the tile products (csrc/gemm_tiles.h), on the CPU: the kernels' own text is compiled for
the host and walked through wave by wave (tests/tiles_check.cpp says what is checked).  A half tile that is asked for again while another
wave may still read it, or read before all of its pieces have arrived, gives wrong sums only when a wave is late, which no
run on a device shows reliably."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def host_form(source: str) -> str:
    """The kernels' text with calls in the place of the assembly, without the launches behind them."""
    source, n = re.subn(r'asm volatile\("s_mov_b32 m0[^;]*;', "sim_fill(base, off, l);", source)
    assert n == 1
    for name, call in ((r"FLLM_VM\(n\)", "sim_vm(n)"), ("FLLM_LGKM0", "sim_lgkm0()")):
        source, n = re.subn(rf"#define {name} asm volatile.*", lambda m: m.group(0).split(" asm ")[0] + " " + call, source)
        assert n == 1
    source = re.sub(r'asm volatile\("" : "\+v"\([^;]*;', ";", source)
    assert "asm" not in source and source.count('#include "common.h"') == 1
    kernels = source.split("// The kernels, products of their own")
    assert len(kernels) == 2
    meeting = re.search(r"^__device__ __forceinline__ bool meet_slices\(.*?^\}$", kernels[1], re.S | re.M).group(0)
    return kernels[0].replace('#include "common.h"', "").replace("#pragma once", "") + "\n" + meeting + "\n}  // namespace fllm_tiles\n"


def test_half_tiles_are_read_after_they_arrive_and_before_they_are_asked_for_again(tmp_path):
    compiler = shutil.which("g++") or shutil.which("clang++")
    if compiler is None:
        pytest.skip("no host C++ compiler")
    with open(os.path.join(ROOT, "fllm_amd", "csrc", "gemm_tiles.h")) as fh:
        (tmp_path / "tiles_host.h").write_text(host_form(fh.read()))
    binary = str(tmp_path / "tiles_check")
    build = subprocess.run([compiler, "-std=c++17", "-O1", "-w", "-I", str(tmp_path), os.path.join(ROOT, "tests", "tiles_check.cpp"), "-o", binary],
                           capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr
    run = subprocess.run([binary], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout + run.stderr
    assert "tiles ok" in run.stdout
