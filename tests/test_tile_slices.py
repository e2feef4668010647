"""Products of many rows whose K several workgroups share: their plan (csrc/plans.h) swept on the CPU under the sanitizers, and the products against float64."""
import os
import shutil
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_plans(tmp_path):
    compiler = shutil.which("g++") or shutil.which("clang++")
    if compiler is None:
        pytest.skip("no host C++ compiler")
    binary = str(tmp_path / "check")
    build = subprocess.run([compiler, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-I",
                            os.path.join(ROOT, "fllm_amd", "csrc"), os.path.join(ROOT, "tests", "tile_slices_check.cpp"), "-o", binary],
                           capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr
    run = subprocess.run([binary], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and "slices ok" in run.stdout, run.stdout + run.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,slices", [(65, 256, 384, 2), (128, 264, 640, 3), (129, 8, 1600, 8), (300, 1000, 576, 3), (513, 2056, 512, 2), (2048, 1536, 384, 2),
                                          (2048, 2048, 8192, 1), (1700, 1536, 13312, 1), (405, 4096, 14336, 1)])
def test_sliced_products(M, N, K, slices):
    """float32 sums of K products of bfloat16 operands that are exact in float64: K 2^-24 of the largest value, below 2^-10; bfloat16 results one rounding
    more (2^-9).  Rows with a stride of their own, last tiles short; from launch to launch no bit differs, whoever comes last."""
    from fllm_amd.kernels import Ops
    ops = Ops()
    gen = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=gen).to(torch.bfloat16).cuda()[:, :K]
    w = (torch.randn(N, K, generator=gen) * K ** -0.5).to(torch.bfloat16).cuda()
    want = x.double() @ w.double().t()
    ops.set_option("linear.tile_slices", slices)
    try:
        made = []
        for _ in range(2):
            f32, b16 = torch.full((M, N), float("nan"), device="cuda"), torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
            assert ops.lib.fllm_linear_tiles(x.data_ptr(), K + 8, w.data_ptr(), None, f32.data_ptr(), N, M, N, K, 1, 0, ops._stream()) == 0
            ops.linear(x, w, b16)
            made.append((f32, b16))
    finally:
        ops.set_option("linear.tile_slices", 1)
    assert (made[0][0].double() - want).abs().max() <= 2.0 ** -10 * want.abs().max()
    assert (made[0][1].double() - want).abs().max() <= 2.0 ** -8 * want.abs().max()
    assert torch.equal(made[0][1], made[0][0].to(torch.bfloat16))
    assert all(torch.equal(a, b) for a, b in zip(*made))
