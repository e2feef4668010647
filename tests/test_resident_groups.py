"""How many workgroups a product of up to 16 rows has (csrc/plans.h), swept on the CPU under the sanitizers, and on the GPU the products where that
number changes, against float64."""
import os
import shutil
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_workgroups_of_every_tile_count(tmp_path):
    compiler = shutil.which("g++") or shutil.which("clang++")
    if compiler is None:
        pytest.skip("no host C++ compiler")
    binary = str(tmp_path / "check")
    build = subprocess.run([compiler, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-I",
                            os.path.join(ROOT, "fllm_amd", "csrc"), os.path.join(ROOT, "tests", "resident_groups_check.cpp"), "-o", binary],
                           capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr
    run = subprocess.run([binary], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and "groups ok" in run.stdout, run.stdout + run.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("tiles,K", [(512, 256), (513, 256), (600, 1536), (768, 264), (769, 256), (1120, 512), (1281, 256)])
def test_gate_up_where_the_number_changes(tiles, K, tiled):
    """A float32 sum of K products of bfloat16 operands (K 2^-24 of the largest), an activation and one rounding (2^-9): under 2^-7 of the largest."""
    from fllm_amd.kernels import Ops
    ops = Ops()
    gen = torch.Generator().manual_seed(tiles)
    inter = 8 * tiles - 3
    w = (torch.randn((2 * inter, K), generator=gen) * K ** -0.5).to(torch.bfloat16).cuda()
    if tiled and not ops.tile_for_decode(w, gate_up=True):
        pytest.skip("a width without copies")
    for M in (1, 8):
        x = torch.randn((M, K), generator=gen).to(torch.bfloat16).cuda()
        y = x.double() @ w.double().t()
        want = torch.nn.functional.silu(y[:, :inter]) * y[:, inter:]
        out = torch.full((M, inter), float("nan"), dtype=torch.bfloat16, device="cuda")
        ops.gate_up_swiglu(x, w, out)
        assert (out.double() - want).abs().max() <= 2.0 ** -7 * want.abs().max()
    ops.forget_copy(w)
