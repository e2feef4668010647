"""Products of 49 to 64 rows around the tiles where the number of their K slices changes (128 to 130, 256 and 257 tiles of 16 columns), every epilogue, with
the tile-major copy and without, against float64: float32 sums of K products of bfloat16 operands (K 2^-24 of the largest, below 2^-10), bfloat16
results one rounding more (2^-9).  From launch to launch, whoever comes last, no bit differs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [49, 64])
@pytest.mark.parametrize("N,K", [(2048, 8192), (2064, 8192), (2080, 8192), (4096, 4096), (4104, 4096)])
def test_every_epilogue(M, N, K):
    from fllm_amd.kernels import Ops
    ops, plain = Ops(), Ops(library_gemm_from=None)
    gen = torch.Generator().manual_seed(M + N + K)
    x = torch.randn((M, K), generator=gen).to(torch.bfloat16).cuda()
    w = (torch.randn((N, K), generator=gen) * K ** -0.5).to(torch.bfloat16).cuda()
    stream, norm, bias = (torch.randn(shape, generator=gen).cuda() for shape in ((M, N), (N,), (N,)))
    y = x.double() @ w.double().t()
    for copy in (False, True):
        if copy and not ops.tile_for_decode(w):
            break
        made = []
        for _ in range(2):
            ops.set_option("linear.slab", 0)
            try:
                f32, b16, res = torch.full_like(stream, float("nan")), torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda"), stream.clone()
                plain.linear(x, w, f32)
                plain.linear(x, w, b16, bias=bias)
                plain.linear(x, w, res, accumulate=True)
                made.append([f32, b16, res])
                if N % 16 == 0:
                    again = stream.clone()
                    prepared = ops.linear_add_prepare(x, w, again, norm)
                    made[-1] += [again, prepared.x, prepared.ssq[:M * prepared.parts]]
            finally:
                ops.set_option("linear.slab", 1)
        assert all(torch.equal(a, b) for a, b in zip(*made))
        f32, b16, res = made[0][:3]
        for got, want, eps in ((f32, y, 2.0 ** -10), (b16, y + bias.double(), 2.0 ** -8), (res, stream.double() + y, 2.0 ** -10)):
            assert (got.double() - want).abs().max() <= eps * want.abs().max()
        if N % 16 == 0:
            want = stream.double() + y
            assert (made[0][3].double() - want).abs().max() <= 2.0 ** -10 * want.abs().max()
            assert (made[0][4].double() - want * norm.double()).abs().max() <= 2.0 ** -8 * (want * norm.double()).abs().max()
            squares = made[0][5].view(M, -1).double().sum(1)
            assert ((squares - (want * want).sum(1)).abs() <= 2.0 ** -9 * squares).all()
    ops.forget_copy(w)
