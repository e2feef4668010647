"""Products of 9 to 16 rows of few tiles and long K, which two workgroups a tile share, against float64: the shortest such K, slices that end inside a
block, one tile, the most tiles and one more, the last tile short.  Sums of K products of bfloat16 operands in float32 (K 2^-24, below 2^-10 here) and, for
bfloat16 results, one rounding (2^-9).  With and without the tile-major copy, and from launch to launch, no bit differs.  Whole (one slice asked for)
and shared they are two orders of the same float32 sum: apart by twice its bound at most."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [8, 9, 13, 16])
@pytest.mark.parametrize("N,K", [(16, 4128), (16, 4104), (1000, 4352), (2048, 4096), (2048, 4224), (2064, 4224), (1536, 13312), (528, 16640)])
def test_sliced_products(M, N, K):
    from fllm_amd.kernels import Ops
    ops = Ops()
    gen = torch.Generator().manual_seed(M + N + K)
    x = torch.randn((M, K), generator=gen).to(torch.bfloat16).cuda()
    w = (torch.randn((N, K), generator=gen) * K ** -0.5).to(torch.bfloat16).cuda()
    stream, norm = torch.randn((M, N), generator=gen).cuda(), (torch.rand(N, generator=gen) + 0.5).cuda()
    y = x.double() @ w.double().t()
    made = []
    for copy in (False, True):
        if copy and not ops.tile_for_decode(w):
            break
        for _ in range(2):
            f32, b16, res = torch.full_like(stream, float("nan")), torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda"), stream.clone()
            ops.linear(x, w, f32)
            ops.linear(x, w, b16)
            outs = [f32, b16, res]
            if N % 16 == 0:
                prepared = ops.linear_add_prepare(x, w, res, norm)
                outs += [prepared.x, prepared.ssq[:M * prepared.parts]]
            else:
                ops.linear(x, w, res, accumulate=True)
            made.append(outs)
    f32, b16, res = made[0][:3]
    assert (f32.double() - y).abs().max() <= 2.0 ** -10 * y.abs().max()
    assert (b16.double() - y).abs().max() <= 2.0 ** -8 * y.abs().max()
    want = stream.double() + y
    assert (res.double() - want).abs().max() <= 2.0 ** -10 * want.abs().max()
    if N % 16 == 0:
        scaled = want * norm.double()
        assert (made[0][3].double() - scaled).abs().max() <= 2.0 ** -8 * scaled.abs().max()
        squares = made[0][4].view(M, -1).double().sum(1)
        assert ((squares - (want * want).sum(1)).abs() <= 2.0 ** -9 * squares).all()
    for other in made[1:]:
        assert all(torch.equal(a, b) for a, b in zip(made[0], other))
    ops.forget_copy(w)


@pytest.mark.parametrize("M", [9, 16])
@pytest.mark.parametrize("N,K", [(16, 4104), (2048, 4224), (1536, 13312)])
def test_whole_where_one_slice_is_asked_for(M, N, K):
    from fllm_amd.kernels import Ops
    ops = Ops()
    gen = torch.Generator().manual_seed(M + N + K)
    x = torch.randn((M, K), generator=gen).to(torch.bfloat16).cuda()
    w = (torch.randn((N, K), generator=gen) * K ** -0.5).to(torch.bfloat16).cuda()
    y, made = x.double() @ w.double().t(), []
    try:
        for slices in (0, 1):
            ops.set_option("linear.slices", slices)
            out = torch.full((M, N), float("nan"), device="cuda")
            made.append(ops.linear(x, w, out))
    finally:
        ops.set_option("linear.slices", 0)
    for out in made:
        assert (out.double() - y).abs().max() <= 2.0 ** -10 * y.abs().max()
    assert (made[0] - made[1]).abs().max() <= 2.0 ** -9 * y.abs().max()
    assert not torch.equal(*made)      # other orders: both forms ran
