"""A row's way into routed experts in one kernel against the kernels that it stands for: the stream and the normed row bit for bit behind a
branch, the picks those of the routers for the row it leaves.  Widths of one to eight steps of 512, one expert, as many as waves, one more, an odd pair of a wave's experts and the
most it takes, both scores, corrections and groups, equal scores, a row that is no number, and what it leaves to the others."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


def operands(rows, width, experts, seed):
    g = torch.Generator().manual_seed(seed)
    draw = lambda *s: torch.randn(*s, generator=g)
    return [t.to(DEV) for t in (draw(rows, width) * 3, draw(rows, width), 1 + 0.3 * draw(width), 1 + 0.3 * draw(width),
                                (draw(experts, width) * 2 * width ** -0.5).to(BF16), torch.rand(experts, generator=g))]


@pytest.mark.parametrize("rows,width,experts,top", [(1, 512, 1, 1), (2, 1536, 8, 2), (5, 1024, 4, 4), (64, 2048, 64, 6), (3, 2560, 6, 3), (7, 4096, 10, 2),
                                                     (4, 512, 9, 2), (2, 1024, 13, 3), (3, 3072, 37, 5)])
@pytest.mark.parametrize("router", ["sigmoid", "softmax", "grouped"])
@pytest.mark.parametrize("behind", ["norm", "scale", "nothing"])
def test_one_kernel_for_sum_norm_and_router(ops, rows, width, experts, top, router, behind):
    x, branch, gain, norm_w, w, correction = operands(rows, width, experts, rows + width)
    if rows > 2:
        w[experts - 1] = w[0]          # equal scores: the lower index
        if behind != "nothing":
            branch[1, 7] = float("nan")
    eps = {"norm": 1e-5, "scale": None, "nothing": None}[behind]
    groups, kept = (2, 1) if experts % 2 == 0 and top <= experts // 2 else (1, 1)
    how = dict(correction=correction, groups=groups, kept=kept) if router == "grouped" else dict(score=router, renormalize=True)

    def route(h):
        ids, weights = torch.empty(rows, top, dtype=torch.int32, device=DEV), torch.empty(rows, top, device=DEV)
        if router == "grouped":
            ops.route_grouped(h, w, correction, top, groups, kept, ids, weights, route_scale=2.5)
            return ids, weights
        ops.route_topk(h, w, top, ids, weights, score=router, renormalize=True, route_scale=2.5)
        return ids, weights

    plain_x, plain_h = x.clone(), torch.empty(rows, width, dtype=BF16, device=DEV)
    if behind == "nothing":
        ops.rmsnorm(plain_x, norm_w, 1e-6, plain_h)
        extra = {}
    else:
        ops.postnorm_add(plain_x, branch, gain, eps, next_weight=norm_w, next_eps=1e-6, next_out=plain_h)
        extra = dict(branch=branch, gain=gain, eps=eps)
    got_x, h = x.clone(), torch.empty(rows, width, dtype=BF16, device=DEV)
    ids, weights = torch.empty(rows, top, dtype=torch.int32, device=DEV), torch.empty(rows, top, device=DEV)
    assert ops.norm_route(got_x, norm_w, 1e-6, h, w, top, ids, weights, route_scale=2.5, **extra, **how)
    same = lambda a, b: torch.equal(a.nan_to_num(12345.0), b.nan_to_num(12345.0))
    assert same(got_x, plain_x)
    if behind == "nothing":      # the norm's factors meet in another order: the neighbouring bfloat16 at most
        assert ((h.float() - plain_h.float()).abs() <= 2.0 ** -7 * plain_h.float().abs()).all()
    else:
        assert same(h, plain_h)
    want_ids, want_weights = route(h)
    assert torch.equal(ids, want_ids) and same(weights, want_weights)


def test_what_it_leaves_to_the_others(ops):
    for rows, width, experts, dtype in ((2, 768, 8, BF16), (65, 512, 8, BF16), (2, 512, 65, BF16), (2, 4608, 8, BF16), (2, 512, 8, torch.float32)):
        x, branch, gain, norm_w, w, _ = operands(rows, width, experts, 1)
        before = x.clone()
        h = torch.full((rows, width), 3.0, dtype=dtype, device=DEV)
        ids, weights = torch.full((rows, 2), -7, dtype=torch.int32, device=DEV), torch.empty(rows, 2, device=DEV)
        assert not ops.norm_route(x, norm_w, 1e-6, h, w.to(dtype), 2, ids, weights, branch=branch, gain=gain, eps=1e-5)
        assert torch.equal(x, before) and bool((h == 3.0).all()) and bool((ids == -7).all())


def test_left_to_the_others_where_plain_kernels_are_asked_for(ops):
    x, _, _, norm_w, w, _ = operands(2, 512, 4, 3)
    before, h = x.clone(), torch.zeros(2, 512, dtype=BF16, device=DEV)
    ids, weights = torch.zeros(2, 1, dtype=torch.int32, device=DEV), torch.zeros(2, 1, device=DEV)
    ops.set_fast_kernels(False)
    try:
        assert not ops.norm_route(x, norm_w, 1e-6, h, w, 1, ids, weights)
    finally:
        ops.set_fast_kernels(True)
    assert torch.equal(x, before) and not h.any() and not weights.any()
