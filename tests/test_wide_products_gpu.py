"""Products of 17 to 128 rows behind a prepared norm, where their pieces end: one to several chunks of columns a slice, sums of squares in
a few to several hundred parts (whole pieces of four and not), row tiles with one live row, matrices whose last tile or row
group is short.  Against float64 on the CPU from the same bfloat16 operands: sums of K products in float32 (K 2^-24, below
2^-11) and one rounding of the result to bfloat16 (2^-9), together under 2^-8 of the largest value; the residual sum stays
float32: 2^-11."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def operands(M, N, K, seed):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn((M, K), generator=gen).to(torch.bfloat16)
    w = (torch.randn((N, K), generator=gen) * K ** -0.5).to(torch.bfloat16)
    return gen, x, w


@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("K,inter,parts", [(1024, 24, 1), (1024, 1000, 3), (2048, 1800, 128), (3072, 520, 260), (4096, 264, 1028)])
def test_scaled_gate_up(M, K, inter, parts):
    from fllm_amd.kernels import Ops, PreparedNorm
    ops = Ops()
    gen, x, w = operands(M, 2 * inter, K, M + K + parts)
    ssq = torch.rand((M, parts), generator=gen) * (2.0 * K / parts) + 1e-3
    scale = 1.0 / torch.sqrt(ssq.double().sum(1, keepdim=True) / K + 1e-5)
    z = x.double() @ w.double().t() * scale
    want = z[:, :inter] / (1 + torch.exp(-z[:, :inter])) * z[:, inter:]
    wd, xd, out = w.cuda(), x.cuda(), torch.empty((M, inter), dtype=torch.bfloat16, device="cuda")
    assert ops.tile_for_decode(wd, gate_up=True)
    prepared = PreparedNorm(xd, ssq.flatten().cuda(), parts)
    ops.norm_gate_up_swiglu(None, None, 1e-5, wd, out, prepared=prepared)
    assert (out.double().cpu() - want).abs().max() <= 2 ** -8 * want.abs().max()
    again = torch.empty_like(out)                # slices are added in their order, whoever comes last
    ops.norm_gate_up_swiglu(None, None, 1e-5, wd, again, prepared=prepared)
    assert torch.equal(out, again)


@pytest.mark.parametrize("M", [17, 33, 48, 49, 65, 128])
@pytest.mark.parametrize("N,K", [(16, 1024), (560, 2048), (2048, 2048), (4096, 4096), (1040, 14336)])
def test_sums_and_the_norm_behind_them(M, N, K):
    from fllm_amd.kernels import Ops
    ops = Ops()
    gen, x, w = operands(M, N, K, M + N + K)
    residual, norm = torch.randn((M, N), generator=gen), torch.rand(N, generator=gen) + 0.5
    bias = torch.randn(N, generator=gen)
    want = residual.double() + x.double() @ w.double().t() + bias.double()
    wd, res = w.cuda(), residual.cuda()
    assert ops.tile_for_decode(wd)
    prepared = ops.linear_add_prepare(x.cuda(), wd, res, norm.cuda(), bias=bias.cuda())
    assert (res.double().cpu() - want).abs().max() <= 2 ** -11 * want.abs().max()
    assert (prepared.x.double().cpu() - want * norm.double()).abs().max() <= 2 ** -8 * (want * norm.double()).abs().max()
    squares = prepared.ssq[:M * prepared.parts].view(M, prepared.parts).double().sum(1).cpu()
    assert ((squares - (want * want).sum(1)).abs() <= 2 ** -10 * squares).all()
