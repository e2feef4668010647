"""Sums and maxima over a wave's lanes (csrc/common.h): their own text compiled for the host, where a value is what all lanes hold (tests/lane_sums_check.cpp
says what is compared), and maxima on the GPU through the softmax of a router's logits: with the largest at every place in turn among values far
below it or of minus infinity, that expert is picked with all of the weight.  exp of 0 is 1 exactly and the others' are 0, so the weights are exact."""
import os
import re
import shutil
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_lanes_meet_as_in_a_butterfly(tmp_path):
    compiler = shutil.which("g++") or shutil.which("clang++")
    if compiler is None:
        pytest.skip("no host C++ compiler")
    with open(os.path.join(ROOT, "fllm_amd", "csrc", "common.h")) as fh:
        text = re.search(r"^struct LanePair \{.*?^__device__ __forceinline__ float wave_max\(float v\) \{.*?^\}$", fh.read(), re.S | re.M).group(0)
    text = re.sub(r"\bunsigned int bits\b", "Lanes bits", text.replace("(int)", ""))
    (tmp_path / "lane_sums_host.h").write_text(re.sub(r"\bfloat\b", "Lanes", text))
    binary = str(tmp_path / "check")
    build = subprocess.run([compiler, "-std=c++17", "-O1", "-I", str(tmp_path), os.path.join(ROOT, "tests", "lane_sums_check.cpp"), "-o", binary],
                           capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr
    run = subprocess.run([binary], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and "lanes ok" in run.stdout, run.stdout + run.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("below", [-float("inf"), -1e30, -200.0])
@pytest.mark.parametrize("experts", [8, 64, 130])
def test_the_largest_logit_at_every_lane(experts, below):
    from fllm_amd.kernels import Ops
    ops = Ops()
    K = 64
    h = torch.zeros((1, K), device="cuda")
    h[0, 0] = 1.0
    for place in range(experts):
        w = torch.zeros((experts, K), device="cuda")
        w[:, 0] = below
        w[place, 0] = -3.0
        ids, weights = torch.full((1, 2), -1, dtype=torch.int32, device="cuda"), torch.full((1, 2), float("nan"), device="cuda")
        ops.route_topk(h, w, 2, ids, weights, score="softmax")
        assert ids[0, 0] == place and weights[0, 0] == 1.0 and weights[0, 1] == 0.0
