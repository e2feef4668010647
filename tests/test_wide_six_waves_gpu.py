"""Products of 17 to 64 rows by workgroups of six waves: with the same K slices they add what workgroups of four add, in the same order, so no bit differs;
row groups that six divides, that end short, and fewer tiles than waves.  Left to the plan, 384 tiles of K 4,096 run as four slices of six waves, and another
shape as the plan likes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def ops():
    from fllm_amd.kernels import Ops
    ops = Ops()
    yield ops
    ops.set_option("linear.wide_waves", 0)
    ops.set_option("linear.slices", 0)


@pytest.mark.parametrize("M", [17, 32, 48, 64])
@pytest.mark.parametrize("heads,kv,d,slices", [(4, 1, 32, 1), (6, 3, 64, 2), (32, 8, 64, 4), (3, 1, 64, 1)])
def test_six_waves_add_as_four(ops, M, heads, kv, d, slices):
    from fllm_amd.kernels import PreparedNorm
    K, page, pages = 2048, 16, 64
    N = (heads + 2 * kv) * d
    gen = torch.Generator().manual_seed(M + N)
    w = (torch.randn((N, K), generator=gen) * K ** -0.5).to(torch.bfloat16).cuda()
    x = torch.randn((M, K), generator=gen).to(torch.bfloat16).cuda()
    prepared = PreparedNorm(x, (torch.rand(M * 128, generator=gen) * 32 + 1e-3).cuda(), 128)
    pos = torch.randint(0, 40, (M,), generator=gen, dtype=torch.int32).cuda()
    seg = torch.arange(M, dtype=torch.int32).cuda()
    tables = torch.randperm(M * 3, generator=gen).to(torch.int32).view(M, 3).cuda()
    cos, sin = torch.randn((64, d // 2), generator=gen).cuda(), torch.randn((64, d // 2), generator=gen).cuda()
    stream = torch.randn((M, N), generator=gen).cuda()
    assert ops.tile_for_decode(w)
    ops.set_option("linear.slices", slices)
    made = []
    for waves in (4, 6):
        ops.set_option("linear.wide_waves", waves)
        q = torch.full((M, heads * d), float("nan"), dtype=torch.bfloat16, device="cuda")
        k = torch.zeros((M * 3, kv, d // 8, page, 8), dtype=torch.bfloat16, device="cuda")
        v = torch.zeros((M * 3, kv, d, page), dtype=torch.bfloat16, device="cuda")
        ops.norm_qkv_rope_store(None, None, 1e-5, w, q, pos, seg, tables, cos, sin, k, v, heads, kv, d, d, page, prepared=prepared)
        added = stream.clone()
        ops.linear(x, w, added, accumulate=True)
        made.append((q, k, v, added))
    assert all(torch.equal(a, b) for a, b in zip(*made))
    want = stream.double() + x.double() @ w.double().t()
    assert (made[1][3].double() - want).abs().max() <= 2.0 ** -11 * want.abs().max()      # float32 sums of K products
    scale = torch.rsqrt(prepared.ssq.view(M, 128).double().sum(1, keepdim=True) / K + 1e-5)
    y = (x.double() @ w.double().t() * scale)[:, :heads * d].view(M, heads, d // 2, 2)
    c, s = cos[pos.long()].double()[:, None], sin[pos.long()].double()[:, None]
    turned = torch.stack((y[..., 0] * c - y[..., 1] * s, y[..., 1] * c + y[..., 0] * s), -1).reshape(M, heads * d)
    assert (made[1][0].double() - turned).abs().max() <= 2.0 ** -8 * turned.abs().max()


@pytest.mark.parametrize("M", [17, 40, 64])
@pytest.mark.parametrize("N,K,slices,waves", [(6144, 4096, 4, 6), (1000, 3072, None, None)])
def test_as_planned(ops, M, N, K, slices, waves):
    gen = torch.Generator().manual_seed(M + N)
    w = (torch.randn((N, K), generator=gen) * K ** -0.5).to(torch.bfloat16).cuda()
    x, stream = torch.randn((M, K), generator=gen).to(torch.bfloat16).cuda(), torch.randn((M, N), generator=gen).cuda()
    assert ops.tile_for_decode(w)
    planned = stream.clone()
    ops.linear(x, w, planned, accumulate=True)
    want = stream.double() + x.double() @ w.double().t()
    assert (planned.double() - want).abs().max() <= 2.0 ** -11 * want.abs().max()
    if slices:
        ops.set_option("linear.slices", slices)
        ops.set_option("linear.wide_waves", waves)
        asked = stream.clone()
        ops.linear(x, w, asked, accumulate=True)
        assert torch.equal(planned, asked)
    ops.forget_copy(w)
