"""Single rows of the two mixers whose keys several workgroups share, put together by the one that counts last: up to 32 shares, rows whose
contexts leave most shares without a key, fewer outputs than threads and more than one trip of them, padding rows, and the same again (the
counters are left at zero)."""
import pytest
import torch

from reference_ops import ReferenceOps
from test_dumizen_gpu import BF16_EPS, DEV, SEGMENTS, SINGLE_ROWS, Scene, close, fill_pools, gen, pooled_attend

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
CONTEXTS = {"long": [(9000, 1), (5, 1), (300, 1)], "many": [(n, 1) for n in (0, 31, 255, 256, 1100, 64, 700, 2300, 511, 12)]}


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


@pytest.mark.parametrize("contexts", ["long", "many"])
@pytest.mark.parametrize("H,G,d,dv", [(1, 1, 32, 32), (16, 1, 64, 128), (12, 2, 128, 128), (9, 3, 96, 64)])
def test_shares_of_single_rows(ops, H, G, d, dv, contexts):
    ref, page, window, pool = ReferenceOps(), 16, 1500, 64
    sc = Scene(CONTEXTS[contexts], G, d, dv, page, seed=H + d, pool=pool)
    g = gen(3)
    q = torch.randn(sc.rows, H * d, generator=g).to(BF16).float()
    r1, r2, pb = torch.rand(H, generator=g) + 0.2, torch.rand(H, generator=g) * 0.5 + 0.05, torch.randn(H, generator=g) - 1.0
    want_t = sc.to("cpu", torch.float64)
    want_t["k_pages"], want_t["v_pages"] = want_t["k_pages"].to(BF16).double(), want_t["v_pages"].to(BF16).double()
    fill_pools(ref, sc, want_t, G, d, dv, pool)
    t = sc.to(DEV, BF16)
    t["pool_k"], t["pool_v"] = want_t["pool_k"].float().to(DEV), want_t["pool_v"].float().to(DEV)

    def sigmoid(o, t, q, kind):
        move = lambda v: v.to(q.device)
        out = torch.full((sc.rows, H * dv), float("nan"), dtype=kind, device=q.device)
        return o.sigmoid_attention(q, t["k_pages"], t["v_pages"], t["tables"], t["row_pos"], t["row_seg"], t["seg_start"], out, H, G, d, dv, page, 0.2, 4.0,
                                   move(r1), move(r2), move(pb), 0.4, 1024, sc.key_chunk, max_context=sc.max_pos)

    pooled_want = pooled_attend(ref, want_t, q.double(), sc, H, G, d, dv, 0.3, window, pool, torch.float64)
    sigmoid_want = sigmoid(ref, want_t, q.double(), torch.float64)
    scale = sigmoid_want.abs().max().item()
    first = None
    for _ in range(3):
        pooled = pooled_attend(ops, t, q.to(DEV, BF16), sc, H, G, d, dv, 0.3, window, pool, BF16)
        weighed = sigmoid(ops, t, q.to(DEV, BF16), BF16)
        close(pooled, pooled_want, 2 * BF16_EPS, 5e-3, "pooled windows")               # the bounds of the attentions' own tests
        close(weighed, sigmoid_want, 2 * BF16_EPS, 4e-3 * scale, "sigmoid weights")
        assert first is None or (torch.equal(pooled, first[0]) and torch.equal(weighed, first[1]))      # whoever counts last adds in one order
        first = (pooled, weighed)
    t["row_seg"][1] = -1                                                               # a padding row of a captured step
    padded = pooled_attend(ops, t, q.to(DEV, BF16), sc, H, G, d, dv, 0.3, window, pool, BF16)
    assert torch.equal(padded[0], first[0][0]) and torch.equal(padded[2:], first[0][2:]) and not padded[1].any()


@pytest.mark.parametrize("rows", ["mixed", "single"])
@pytest.mark.parametrize("H,G,d,dv,page,pool", [(4, 1, 32, 64, 48, 8), (8, 2, 64, 96, 48, 20), (9, 3, 96, 96, 48, 16), (12, 2, 128, 128, 80, 32)])
def test_pages_that_are_no_power_of_two(ops, H, G, d, dv, page, pool, rows):
    """Pages of a power of two have instances of their own; these are the others, with blocks that divide the pages and blocks that do not."""
    ref, window = ReferenceOps(), 70
    sc = Scene(SINGLE_ROWS if rows == "single" else SEGMENTS, G, d, dv, page, seed=H + d, pool=pool)
    g = gen(3)
    q = torch.randn(sc.rows, H * d, generator=g).to(BF16).float()
    r1, r2, pb = torch.rand(H, generator=g) + 0.2, torch.rand(H, generator=g) * 0.5 + 0.05, torch.randn(H, generator=g) - 1.0
    want_t = sc.to("cpu", torch.float64)
    want_t["k_pages"], want_t["v_pages"] = want_t["k_pages"].to(BF16).double(), want_t["v_pages"].to(BF16).double()
    fill_pools(ref, sc, want_t, G, d, dv, pool)
    t = sc.to(DEV, BF16)
    t["pool_k"], t["pool_v"] = want_t["pool_k"].float().to(DEV), want_t["pool_v"].float().to(DEV)
    outs = []
    for o, tensors, on, kind in ((ref, want_t, "cpu", torch.float64), (ops, t, DEV, BF16)):
        pooled = pooled_attend(o, tensors, q.to(on, kind), sc, H, G, d, dv, 0.3, window, pool, kind)
        weighed = torch.empty(sc.rows, H * dv, dtype=kind, device=on)
        o.sigmoid_attention(q.to(on, kind), tensors["k_pages"], tensors["v_pages"], tensors["tables"], tensors["row_pos"], tensors["row_seg"],
                            tensors["seg_start"], weighed, H, G, d, dv, page, 0.2, 4.0, r1.to(on), r2.to(on), pb.to(on), 0.4, 8, sc.key_chunk,
                            max_context=sc.max_pos)
        outs.append((pooled, weighed))
    close(outs[1][0], outs[0][0], 2 * BF16_EPS, 5e-3, "pooled windows")                # the bounds of the attentions' own tests
    close(outs[1][1], outs[0][1], 2 * BF16_EPS, 4e-3 * outs[0][1].abs().max().item(), "sigmoid weights")
