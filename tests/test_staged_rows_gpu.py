"""How products of up to 16 rows lay their rows out in LDS, where the pieces end: a wave's range of 64 to 128 columns (four rows a load), to 256 (two) and
more, short last ranges and waves without one, rows that fill a load, a batch of four and one more.  Against float64: float32 sums of K products (K 2^-24),
an activation and one rounding to bfloat16 (2^-9), under 2^-7 of the largest value; behind a norm the rows are rounded to bfloat16 first (2^-9 each, of
random sign): the same bound."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [72, 256, 1000, 1024, 1536, 2048, 2056, 2560, 4096])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 7, 8, 9, 15, 16])
def test_staged_rows(M, K):
    from fllm_amd.kernels import Ops
    ops = Ops()
    gen = torch.Generator().manual_seed(100 * M + K)
    inter = 520
    wide = torch.randn((M, K + 8), generator=gen).cuda()
    x, norm = wide[:, :K].contiguous(), (torch.rand(K, generator=gen) + 0.5).cuda()
    rows = wide.to(torch.bfloat16)[:, :K]                     # a row stride of its own
    w = (torch.randn((2 * inter, K), generator=gen) * K ** -0.5).to(torch.bfloat16).cuda()
    assert K % 32 or K < 256 or ops.tile_for_decode(w, gate_up=True)

    def gated(y):
        return torch.nn.functional.silu(y[:, :inter]) * y[:, inter:]

    out = torch.full((M, inter), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.gate_up_swiglu(rows, w, out)
    want = gated(rows.double() @ w.double().t())
    assert (out.double() - want).abs().max() <= 2.0 ** -7 * want.abs().max()
    normed = x.double() * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5) * norm.double()
    want = gated(normed @ w.double().t())
    ops.norm_gate_up_swiglu(x, norm, 1e-5, w, out.fill_(float("nan")))
    assert (out.double() - want).abs().max() <= 2.0 ** -7 * want.abs().max()
    ops.forget_copy(w)
