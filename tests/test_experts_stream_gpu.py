"""Routed experts of decode steps from their tile-major copies (`Ops.experts_stream`), against the float64 products of the same
operands: column tiles that the matrices fill partly, waves without a product of their own, more pairs of an expert than one and
than two groups of 16, experts without a pair, fewer pairs than experts, ids outside the stack, and what is declined."""
import pytest
import torch

from reference_ops import ReferenceOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16_EPS = 2.0 ** -8


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


@pytest.mark.parametrize("spread", ["random", "one expert"])
@pytest.mark.parametrize("gated,weighted,limit,alpha,offset", [(True, True, 0.0, 1.0, 0.0), (True, False, 1.5, 1.702, 1.0), (False, False, 0.0, 1.0, 0.0)])
@pytest.mark.parametrize("rows,width,inter,experts,top", [(1, 256, 256, 8, 2), (3, 288, 320, 9, 1), (8, 1536, 480, 8, 2), (17, 512, 288, 3, 2),
                                                          (64, 256, 256, 8, 2), (40, 272 + 16, 256, 5, 2), (128, 256, 288, 32, 4), (2, 1024, 256, 8, 2),
                                                          (9, 1312, 256, 8, 2), (3, 2560, 288, 8, 2)])
def test_the_picked_experts_stream_from_their_copies(ops, rows, width, inter, experts, top, gated, weighted, limit, alpha, offset, spread):
    ref = ReferenceOps()
    g = torch.Generator().manual_seed(rows * 31 + width)
    dtype = torch.bfloat16
    h = torch.randn(rows, width, generator=g).to(dtype)
    n_up = (2 if gated else 1) * inter
    w_up = (torch.randn(experts, n_up, width, generator=g) * 2 * width ** -0.5).to(dtype).to(DEV)
    w_down = (torch.randn(experts, width, inter, generator=g) * inter ** -0.5).to(dtype).to(DEV)
    ids = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(rows)]).to(torch.int32)
    if spread == "one expert":
        ids[:, 0] = experts - 1
    weights = torch.rand(rows, top, generator=g)
    args = (h.to(DEV), ids.to(DEV), weights.to(DEV) if weighted else None, w_up, w_down)
    out = torch.full((rows * top, width), float("nan"), dtype=torch.float32, device=DEV)
    assert not ops.experts_stream(*args, out, gated, limit, alpha, offset) and out.isnan().all()      # no copies yet
    assert ops.tile_experts(w_up) and ops.tile_experts(w_down)
    taken = ops.experts_stream(*args, out, gated, limit, alpha, offset)
    assert taken == (rows * top <= 16 * experts)
    if not taken:
        return
    want_act = torch.empty(rows * top, inter, dtype=torch.float64)
    if gated:
        ref.experts_gate_up(h, ids, weights if weighted else torch.ones(rows, top), w_up.cpu(), want_act, limit, alpha, offset)
    else:
        ref.experts_up(h, ids, w_up.cpu(), want_act)
    want = torch.empty(rows * top, width, dtype=torch.float64)
    ref.experts_down(want_act.to(dtype), ids, w_down.cpu(), want)
    # one rounding of the scaled rows and one of the activations, as the grouped kernel's test allows
    assert ((out.cpu().double() - want).abs() <= 2 * BF16_EPS * (want.abs() + want.abs().max())).all()
    # a pair's bits do not depend on the rows beside it
    keep = torch.arange(rows)[rows // 2:]
    part = torch.empty(len(keep) * top, width, dtype=torch.float32, device=DEV)
    assert ops.experts_stream(args[0][keep], args[1][keep].contiguous(), args[2][keep].contiguous() if weighted else None, w_up, w_down, part, gated, limit,
                              alpha, offset)
    assert torch.equal(part, out.view(rows, top, width)[keep.to(DEV)].reshape(-1, width))
    # ids outside the stack read its first and last expert, as in the plain kernels
    wild, tame = ids.clone(), ids.clone()
    wild[0, 0], tame[0, 0] = experts + 5, experts - 1
    wild[-1, -1], tame[-1, -1] = -3, 0
    a, b = torch.empty_like(out), torch.empty_like(out)
    assert ops.experts_stream(args[0], wild.to(DEV), args[2], w_up, w_down, a, gated, limit, alpha, offset)
    assert ops.experts_stream(args[0], tame.to(DEV), args[2], w_up, w_down, b, gated, limit, alpha, offset)
    assert torch.equal(a, b)


def test_what_has_no_copy_and_what_is_declined(ops):
    for shape, dtype in (((4, 24, 256), torch.bfloat16), ((4, 32, 264), torch.bfloat16), ((4, 32, 128), torch.bfloat16), ((4, 32, 256), torch.float32)):
        assert not ops.tile_experts(torch.zeros(shape, dtype=dtype, device=DEV))
    w = torch.randn(2, 512, 256, device=DEV).to(torch.bfloat16)
    d = torch.randn(2, 256, 512, device=DEV).to(torch.bfloat16)
    assert ops.tile_experts(w) and ops.tile_experts(d)
    h, ids, out = torch.randn(2, 256, device=DEV).to(torch.bfloat16), torch.zeros(2, 1, dtype=torch.int32, device=DEV), torch.empty(2, 256, device=DEV)
    ops.set_fast_kernels(False)
    try:
        assert not ops.experts_stream(h, ids, None, w, d, out, gated=False)
    finally:
        ops.set_fast_kernels(True)
    assert ops.experts_stream(h, ids, None, w, d, out, gated=False)
    key = w.data_ptr()
    del w
    assert key not in type(ops)._tiles                       # the copy goes with its stack
