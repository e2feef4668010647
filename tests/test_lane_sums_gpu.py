"""Sums over the lanes of a wave: a row with one value that is not zero, at every place of the row in turn, is normed to the root of the width (times the
weight) wherever it stands; a lane that counted twice or not at all would show as a factor of the root of two, or as infinity.  The sum is exact (one
square and zeros); what follows is a division, a root and two products in float32: 2^-21."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [8, 64, 136, 512, 1536])
def test_every_lane_counts_once(width):
    from fllm_amd.kernels import Ops
    ops = Ops()
    gen = torch.Generator().manual_seed(width)
    value = torch.rand(width, generator=gen) + 0.5
    x = torch.diag(value).cuda()
    weight = (torch.rand(width, generator=gen) + 0.5).cuda()
    out = torch.full((width, width), float("nan"), device="cuda")
    ops.rmsnorm(x, weight, 1e-30, out)
    want = torch.diag(weight.double() * width ** 0.5)
    assert ((out.double() - want).abs() <= 2.0 ** -21 * want).all()


@pytest.mark.parametrize("rows,K", [(1, 256), (4, 1536), (16, 2048), (16, 4096)])
def test_every_lane_counts_once_in_a_product(rows, K):
    """The norm inside a product, a one at another place in every row: 64 of K places, among them the ends of all waves' ranges; the product of one
    bfloat16 operand is exact, the row's scale is a float32 root, and the result is rounded to bfloat16 (2^-9)."""
    from fllm_amd.kernels import Ops
    ops = Ops()
    w = torch.ones((16, K), dtype=torch.bfloat16, device="cuda")
    out = torch.empty((rows, 16), dtype=torch.bfloat16, device="cuda")
    places = sorted({0, 1, K - 1, K // 2, K // 2 - 1} | {i * K // 60 for i in range(60)})
    for at in range(0, len(places), rows):
        x = torch.zeros((rows, K), device="cuda")
        for r in range(rows):
            x[r, places[(at + r) % len(places)]] = 1.0
        ops.norm_linear(x, torch.ones(K, device="cuda"), 1e-30, w, out)
        assert (out.float() - K ** 0.5).abs().max() <= 2.0 ** -8 * K ** 0.5
