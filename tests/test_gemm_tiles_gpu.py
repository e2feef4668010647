"""Products of many rows on 256- and 128-row tiles (gemm_tiles.h) against float64: tiles of one row, rows and columns that no tile divides,
the shortest K, K of an odd number of steps (128-row tiles), more tiles than workgroups for each row tile and epilogue, and grouped by expert
with experts of no pair, one pair and several tiles, and with more tiles than workgroups in both products.  Tolerance: operands are exact in float64, so an output may be off by the float32 sum (K * 2^-24 of the
sum of the products' sizes, which random signs keep far below) and one rounding to bfloat16, 2^-9; twice that, of the value and of a
hundredth of the largest."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16_EPS = 2.0 ** -8


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


def close(got, want, eps):
    want = want.to(got.device)
    off = (got.double() - want).abs()
    assert (off <= eps * (want.abs() + 0.01 * want.abs().max())).all(), (off / (want.abs() + 0.01 * want.abs().max())).max()


def ptr(t):
    return None if t is None else t.data_ptr()


@pytest.mark.parametrize("bm", [128, 256])
@pytest.mark.parametrize("M,N,K", [(1, 8, 256), (129, 264, 256), (300, 520, 384), (257, 4104, 512), (2304, 1288, 256), (1500, 5000, 768)])
def test_every_epilogue(ops, M, N, K, bm):
    g = torch.Generator().manual_seed(M + N)
    wide = torch.randn(M, K + 8, generator=g).to(torch.bfloat16).to(DEV)
    x = wide[:, :K]                                             # a row stride of its own
    w = (torch.randn(2 * N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    y = x.double() @ w.double().T
    first = y[:, :N]
    stream = ops._stream()
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    for limit, alpha, offset in ((0.0, 1.0, 0.0), (0.7, 1.702, 1.0)):
        assert ops.lib.fllm_gate_up_tiles(ptr(x), K + 8, ptr(w), ptr(out), M, N, K, limit, alpha, offset, bm, stream) == 0
        gate, up = (first.clamp(max=limit), y[:, N:].clamp(-limit, limit)) if limit else (first, y[:, N:])
        close(out, gate * torch.sigmoid(alpha * gate) * (up + offset), 2 * BF16_EPS)
    for mode, b, want in ((0, None, first), (0, bias, first + bias.double()), (2, None, first.clamp(min=0) ** 2)):
        out.fill_(float("nan"))
        assert ops.lib.fllm_linear_tiles(ptr(x), K + 8, ptr(w), ptr(b), ptr(out), N, M, N, K, mode, bm, stream) == 0
        close(out, want, BF16_EPS)
    beside = torch.full((M, N + 16), float("nan"), dtype=torch.bfloat16, device=DEV)     # columns beside the output stay as they are
    assert ops.lib.fllm_linear_tiles(ptr(x), K + 8, ptr(w), None, ptr(beside), N + 16, M, N, K, 0, bm, stream) == 0
    close(beside[:, :N], first, BF16_EPS)
    assert beside[:, N:].isnan().all()


@pytest.mark.parametrize("bm,K", [(256, 256), (256, 640), (128, 192), (128, 448)])
def test_workgroups_that_take_several_tiles(ops, bm, K):
    """A launch has 256 workgroups at most.  2,100 rows x 8,200 columns are 297 tiles of 256 rows (gate and up 585), 561 of 128 (1,105): a workgroup
    asks for its next tile's first steps before it stores the one that it has, and the last row and column tiles are ragged."""
    M, N = 2100, 8200
    g = torch.Generator().manual_seed(K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(2 * N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    y = x.double() @ w.double().T
    gate, up = y[:, :N], y[:, N:]
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert ops.lib.fllm_gate_up_tiles(ptr(x), K, ptr(w), ptr(out), M, N, K, 0.0, 1.0, 0.0, bm, ops._stream()) == 0
    close(out, gate * torch.sigmoid(gate) * up, 2 * BF16_EPS)
    for mode, b, want in ((0, None, gate), (0, bias, gate + bias.double()), (2, None, gate.clamp(min=0) ** 2)):
        out.fill_(float("nan"))
        assert ops.lib.fllm_linear_tiles(ptr(x), K, ptr(w), ptr(b), ptr(out), N, M, N, K, mode, bm, ops._stream()) == 0
        close(out, want, BF16_EPS)


@pytest.mark.parametrize("M,N,K", [(200, 264, 192), (140, 1032, 320)])
def test_an_odd_number_of_steps(ops, M, N, K):
    g = torch.Generator().manual_seed(K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    assert ops.lib.fllm_linear_tiles(ptr(x), K, ptr(w), None, ptr(out), N, M, N, K, 0, 1, ops._stream()) == 0
    close(out, x.double() @ w.double().T, BF16_EPS)


def test_what_is_declined(ops):
    x = torch.zeros(256, 256, dtype=torch.bfloat16, device=DEV)
    out = torch.empty(256, 256, dtype=torch.bfloat16, device=DEV)
    linear = lambda *a: ops.lib.fllm_linear_tiles(*a, ops._stream())
    assert linear(ptr(x), 256, ptr(x), None, ptr(out), 256, 256, 252, 256, 0, 1) == 1      # columns in eights
    assert linear(ptr(x), 256, ptr(x), None, ptr(out), 256, 256, 256, 128, 0, 1) == 1      # three steps of 64 at least
    assert linear(ptr(x), 256, ptr(x), None, ptr(out), 256, 256, 128, 224, 0, 1) == 1      # whole steps
    assert linear(ptr(x) + 2, 256, ptr(x), None, ptr(out), 256, 200, 128, 192, 0, 1) == 1  # operands on 16 bytes
    assert linear(ptr(x), 256, ptr(x), None, ptr(out), 256, 256, 256, 256, 0, 0) == 1      # a quarter of a round: left to the library
    for width, asked in ((192, 256), (128, 128), (256, 2), (256, 192), (256, -1)):         # a row tile that cannot walk this K; no row tile
        assert linear(ptr(x), 256, ptr(x), None, ptr(out), 256, 200, 128, width, 0, asked) == 1
        assert ops.lib.fllm_gate_up_tiles(ptr(x), 256, ptr(x), ptr(out), 200, 128, width, 0.0, 1.0, 0.0, asked, ops._stream()) == 1
    assert not ops.gate_up_tiles(x[:64], x, out[:64, :128].contiguous())
    assert ops.gate_up_tiles(x[:65], x, out[:65, :128].contiguous())


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("rows,width,inter,experts,top,spread", [(400, 256, 256, 8, 2, "random"), (1200, 256, 384, 5, 2, "uneven"), (300, 512, 256, 3, 1, "one")])
def test_experts_on_large_tiles(ops, rows, width, inter, experts, top, spread, gated):
    g = torch.Generator().manual_seed(rows)
    bf = torch.bfloat16
    h = torch.randn(rows, width, generator=g).to(bf)
    w_up = (torch.randn(experts, (2 if gated else 1) * inter, width, generator=g) * 2 * width ** -0.5).to(bf)
    w_down = (torch.randn(experts, width, inter, generator=g) * inter ** -0.5).to(bf)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(rows)]).to(torch.int32)
    if spread == "uneven":                                      # an expert of one pair, one of none, the others of several tiles
        ids = torch.stack([torch.randperm(experts - 2, generator=g)[:top] for _ in range(rows)]).to(torch.int32)
        ids[7, 1] = experts - 1
    elif spread == "one":
        ids[:] = 1
    weights = torch.rand(rows, top, generator=g)
    assert rows * top // experts >= 96
    out = torch.full((rows * top, width), float("nan"), device=DEV)
    if gated:
        assert ops.experts_grouped(h.to(DEV), ids.to(DEV), weights.to(DEV), w_up.to(DEV), w_down.to(DEV), out)
    else:
        assert ops.experts_grouped_ungated(h.to(DEV), ids.to(DEV), w_up.to(DEV), w_down.to(DEV), out)
    want = torch.empty(rows * top, width, dtype=torch.float64)
    flat = ids.reshape(-1).long()
    for e in range(experts):
        at = torch.nonzero(flat == e).flatten()
        x = h[at // top]
        if gated:
            x = (x.float() * weights.reshape(-1)[at][:, None]).to(bf)
        y = x.double() @ w_up[e].double().T
        act = torch.nn.functional.silu(y[:, :inter]) * y[:, inter:] if gated else y.clamp(min=0) ** 2
        want[at] = act.to(bf).double() @ w_down[e].double().T
    # an activation whose float32 sum lies next to a rounding boundary may round the other way: its step of 2^-8, times its weight, is below
    # two steps of the largest output (the largest activation times the largest weight is below twice that output)
    off = (out.cpu().double() - want).abs()
    assert (off <= 2 * BF16_EPS * (want.abs() + want.abs().max())).all() and off.norm() <= 1e-3 * want.norm()


@pytest.mark.parametrize("gated,inter", [(True, 2048), (False, 4096)])
@pytest.mark.parametrize("rows", [3000, 3840])      # tiles of 128 rows and of 256 take fewer rounds
def test_experts_with_more_tiles_than_workgroups(ops, rows, gated, inter):
    """6,000 and 7,680 pairs of four experts: 300 to 800 tiles in either product, the last of an expert ragged."""
    g = torch.Generator().manual_seed(rows)
    bf, experts, top, width = torch.bfloat16, 4, 2, 3072
    h = torch.randn(rows, width, generator=g).to(bf).to(DEV)
    w_up = (torch.randn(experts, (2 if gated else 1) * inter, width, generator=g) * 2 * width ** -0.5).to(bf).to(DEV)
    w_down = (torch.randn(experts, width, inter, generator=g) * inter ** -0.5).to(bf).to(DEV)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(rows)]).to(torch.int32).to(DEV)
    weights = torch.rand(rows, top, generator=g).to(DEV)
    out = torch.full((rows * top, width), float("nan"), device=DEV)
    if gated:
        assert ops.experts_grouped(h, ids, weights, w_up, w_down, out)
    else:
        assert ops.experts_grouped_ungated(h, ids, w_up, w_down, out)
    flat = ids.reshape(-1).long()
    for e in range(experts):
        at = torch.nonzero(flat == e).flatten()
        x = h[at // top]
        if gated:
            x = (x.float() * weights.reshape(-1)[at][:, None]).to(bf)
        y = x.double() @ w_up[e].double().T
        act = torch.nn.functional.silu(y[:, :inter]) * y[:, inter:] if gated else y.clamp(min=0) ** 2
        want = act.to(bf).double() @ w_down[e].double().T
        off = (out[at].double() - want).abs()               # the bound of the test above
        assert (off <= 2 * BF16_EPS * (want.abs() + want.abs().max())).all() and off.norm() <= 1e-3 * want.norm()
