"""Products of 256-row tiles whose last round runs as tiles of half the rows, against float64: no whole round before the halves, one and more; last row
tiles of one row, of 128, of 129 (a second half of no row, of one); every epilogue, and grouped by expert.  Tolerance: as in
test_gemm_tiles_gpu.py, operands are exact in float64, so an output may be off by its float32 sum and one rounding to bfloat16, 2^-9; twice that,
of the value and of a hundredth of the largest.  A tile's sums are the same whole or in halves: with and without them no bit differs."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16_EPS = 2.0 ** -8


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    ops = Ops()
    yield ops
    ops.set_option("linear.half_tiles", 1)


def close(got, want, eps):
    off = (got.double() - want).abs()
    assert (off <= eps * (want.abs() + 0.01 * want.abs().max())).all(), (off / (want.abs() + 0.01 * want.abs().max())).max()


@pytest.mark.parametrize("M,N,K", [(1, 264, 256), (129, 520, 384), (384, 8200, 256), (1025, 16392, 256), (2177, 8712, 512), (2100, 16400, 256)])
def test_every_epilogue(ops, M, N, K):
    g = torch.Generator().manual_seed(M + N)
    wide = torch.randn(M, K + 8, generator=g).to(torch.bfloat16).to(DEV)
    x = wide[:, :K]
    w = (torch.randn(2 * N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    y = x.double() @ w.double().T
    gate, up = y[:, :N], y[:, N:]
    made = {}
    for halves in (0, 2):
        ops.set_option("linear.half_tiles", halves)
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        assert ops.lib.fllm_gate_up_tiles(x.data_ptr(), K + 8, w.data_ptr(), out.data_ptr(), M, N, K, 0.0, 1.0, 0.0, 256, ops._stream()) == 0
        close(out, gate * torch.sigmoid(gate) * up, 2 * BF16_EPS)
        made[halves] = [out]
        for mode, b, want in ((0, bias, gate + bias.double()), (0, None, gate), (2, None, gate.clamp(min=0) ** 2)):
            out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
            assert ops.lib.fllm_linear_tiles(x.data_ptr(), K + 8, w.data_ptr(), None if b is None else b.data_ptr(), out.data_ptr(), N, M, N, K, mode, 256, ops._stream()) == 0
            close(out, want, BF16_EPS)
            made[halves].append(out)
    assert all(torch.equal(a, b) for a, b in zip(made[0], made[2]))


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("rows,experts,inter,width", [(1024, 4, 1024, 1024), (1900, 8, 4480, 512), (1029, 2, 3072, 3072)])
def test_experts(ops, rows, experts, inter, width, gated):
    """Counts that the row tiles are chosen by in the entry point; whether halves run is up to the tiles that the pairs fill."""
    g = torch.Generator().manual_seed(rows)
    bf, top = torch.bfloat16, 2
    h = torch.randn(rows, width, generator=g).to(bf).to(DEV)
    w_up = (torch.randn(experts, (2 if gated else 1) * inter, width, generator=g) * 2 * width ** -0.5).to(bf).to(DEV)
    w_down = (torch.randn(experts, width, inter, generator=g) * inter ** -0.5).to(bf).to(DEV)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(rows)]).to(torch.int32).to(DEV)
    made = []
    for halves in (0, 1):
        ops.set_option("linear.half_tiles", halves)
        out = torch.full((rows * top, width), float("nan"), device=DEV)
        if gated:
            assert ops.experts_grouped(h, ids, None, w_up, w_down, out)
        else:
            assert ops.experts_grouped_ungated(h, ids, w_up, w_down, out)
        made.append(out)
    assert torch.equal(*made)
    flat = ids.reshape(-1).long()
    for e in range(experts):
        at = torch.nonzero(flat == e).flatten()
        y = h[at // top].double() @ w_up[e].double().T
        act = torch.nn.functional.silu(y[:, :inter]) * y[:, inter:] if gated else y.clamp(min=0) ** 2
        want = act.to(bf).double() @ w_down[e].double().T
        # an activation that rounds the other way: its step of 2^-8 times its weight is below two steps of the largest output
        off = (made[0][at].double() - want).abs()
        assert (off <= 2 * BF16_EPS * (want.abs() + want.abs().max())).all() and off.norm() <= 1e-3 * want.norm()
