"""Decode steps of experts without a gate beside a shared expert, one stream of weights a product (`experts_stream_shared`), against float64:
a row to as many as one pass takes, one to three picks, few experts and more than there are pairs, a shared expert narrower and wider than
the others, widths whose last wave has less than the others and column counts that end inside a workgroup's columns."""
import pytest
import torch

from fllm_amd.config.spec import PartSpec
from fllm_amd.registry import part_class

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


def draw(shape, seed, scale):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(BF16).to(DEV)


def reference(h, ids, weights, up, down, shared_up, shared_down):
    h = h.double()
    act = torch.einsum("rtik,rk->rti", up.double()[ids.long()], h).clamp(min=0) ** 2
    parts = torch.einsum("rtni,rti->rtn", down.double()[ids.long()], act.to(BF16).double()) * weights.double()[:, :, None]
    common = ((h @ shared_up.double().T).clamp(min=0) ** 2).to(BF16).double() @ shared_down.double().T
    return torch.cat([parts, common[:, None]], 1).flatten(0, 1)


@pytest.mark.parametrize("rows,top,E,inter,shared,K", [(1, 1, 4, 256, 512, 256), (1, 2, 8, 4480, 4480, 1536), (2, 2, 8, 288, 256, 544), (5, 3, 70, 256, 1056, 320),
                                                       (16, 3, 8, 544, 288, 1536), (16, 1, 1, 256, 256, 288), (13, 2, 8, 2048, 4096, 1024)])
def test_stream_with_a_shared_expert(ops, rows, top, E, inter, shared, K):
    g = torch.Generator().manual_seed(rows + E)
    h = draw((rows, K), 1, 1.0)
    up, down = draw((E, inter, K), 2, K ** -0.5), draw((E, K, inter), 3, inter ** -0.5)
    shared_up, shared_down = draw((shared, K), 4, K ** -0.5), draw((K, shared), 5, shared ** -0.5)
    ids = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(rows)]).int().to(DEV)
    weights = torch.rand(rows, top, generator=g).to(DEV)
    out = torch.full((rows * (top + 1), K), float("nan"), device=DEV)
    assert not ops.experts_stream_shared(h, ids, weights, up, down, shared_up, shared_down, out)       # no copies yet
    assert ops.tile_experts(up) and ops.tile_experts(down) and ops.tile_for_decode(shared_up) and ops.tile_for_decode(shared_down)
    ops.set_fast_kernels(False)
    try:
        assert not ops.experts_stream_shared(h, ids, weights, up, down, shared_up, shared_down, out) and out.isnan().all()
    finally:
        ops.set_fast_kernels(True)
    assert ops.experts_stream_shared(h, ids, weights, up, down, shared_up, shared_down, out)
    want = reference(h, ids, weights, up, down, shared_up, shared_down)
    # an activation may round to the neighbouring bfloat16, 2^-8 of it: a sum of `inter` terms with signs of their own is off by no more
    # than about 2^-8 of itself
    bound = 2.0 ** -8 * want.abs().max().item()
    assert (out.double() - want).abs().max().item() <= bound


def test_more_rows_than_one_pass_takes_are_left_to_the_others(ops):
    up, down, shared_up, shared_down = draw((8, 256, 256), 2, 0.1), draw((8, 256, 256), 3, 0.1), draw((256, 256), 4, 0.1), draw((256, 256), 5, 0.1)
    for w in (up, down):
        assert ops.tile_experts(w)
    for w in (shared_up, shared_down):
        assert ops.tile_for_decode(w)
    assert ops.experts_stream_shared_takes(16, 3, up, down, shared_up, shared_down)
    assert not ops.experts_stream_shared_takes(17, 2, up, down, shared_up, shared_down)
    assert not ops.experts_stream_shared_takes(2, 4, up, down, shared_up, shared_down)


@pytest.mark.parametrize("rows", [1, 16, 17])
def test_the_part_leaves_what_its_plain_kernels_sum_to(ops, rows):
    from fllm_amd.parts.runtime import Runtime
    rt = Runtime(torch.device(DEV), BF16, ops, 64, decode_weight_tiles=True)
    params = dict(hidden_size=320, intermediate_size=256, experts=4, top=2, score="sigmoid", renormalize=True, weight_on="output", gated=False,
                  route_scale=2.5, shared=288, groups=2, groups_kept=1)
    names = ["router", "correction", "shared_up", "shared_down"] + [f"{k}_{e}" for k in ("up", "down") for e in range(4)]
    cls = part_class("feed_forward", "routed_experts")
    shapes = cls.tensor_shapes(params)
    w = {n: draw(shapes[n][0], i, 0.06) for i, n in enumerate(names)}
    part = cls(PartSpec("routed_experts", params, {n: n for n in names}), w, rt)
    h = draw((rows, 320), 77, 1.0)
    parts = part.branch_parts_for(rows)
    assert parts == (3 if rows <= 16 else 1)
    branch = torch.full((rows * parts, 320), float("nan"), device=DEV)
    part.forward(None, h, None, branch=branch)
    ops.set_fast_kernels(False)
    try:
        plain = torch.full((rows * parts, 320), float("nan"), device=DEV)
        part.forward(None, h, None, branch=plain)
    finally:
        ops.set_fast_kernels(True)
    got, want = branch.view(rows, parts, 320).sum(1), plain.view(rows, parts, 320).sum(1)
    # both round the activations to bfloat16 (2^-9 each) from sums in another order
    assert (got - want).abs().max() <= 2.0 ** -7 * want.abs().max()
