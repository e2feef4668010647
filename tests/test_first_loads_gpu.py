"""The forms of small kernels that ask for everything at once, where a rule sends a call to one or the other: each against the form beside it, which
does the same arithmetic in the same order, so that the bits are the same; and the picks of routers, against a sort on the host."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F32, BF16 = torch.float32, torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


def off(t):
    """A dense copy of t that begins one element behind a 16-byte boundary."""
    out = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    return out.copy_(t)


def picks(choice, top):
    """The `top` largest in turn, the lower index among equals; where nothing compares, expert k."""
    left, out = list(choice), []
    for k in range(top):
        best = [e for e, c in enumerate(left) if c == c and c > -float("inf")]
        at = max(best, key=lambda e: (left[e], -e)) if best else k
        out.append(at)
        left[at] = -float("inf")
    return out


@pytest.mark.parametrize("experts,top,groups,kept", [(1, 1, 1, 1), (8, 2, 4, 2), (12, 5, 3, 2), (63, 6, 1, 1), (64, 8, 64, 9), (64, 64, 1, 1), (65, 8, 5, 3), (128, 7, 8, 2)])
@pytest.mark.parametrize("nan", [False, True])
def test_picks_of_equals_and_of_rows_that_compare_with_nothing(ops, experts, top, groups, kept, nan):
    """Scores from nine values, so that most are equals; 64 experts are a wave's lanes.  A row picks the logit its one lane names."""
    g = torch.Generator().manual_seed(experts)
    rows, K = 4, 64
    w = (torch.randint(-4, 5, (experts, K), generator=g) * 0.5).to(BF16)
    h = torch.zeros(rows, K, dtype=BF16)
    for r in range(rows):
        h[r, r] = 1.0
    if nan:
        h[rows - 1, 0] = float("nan")
    z = h.float() @ w.float().T
    z[(h != h).any(1)] = float("nan")
    ids, weights = torch.empty(rows, top, dtype=torch.int32, device=DEV), torch.empty(rows, top, device=DEV)
    ops.route_topk(h.to(DEV), w.to(DEV), top, ids, weights)
    want = [picks(z[r].tolist(), top) for r in range(rows)]      # the sigmoid rises
    assert ids.cpu().tolist() == want
    score = torch.sigmoid(z.double())
    torch.testing.assert_close(weights[:3].double().cpu(), torch.stack([score[r][want[r]] for r in range(3)]), rtol=1e-6, atol=1e-7)
    correction = torch.randint(0, 3, (experts,), generator=g) * 0.25
    ids2, weights2 = torch.empty_like(ids), torch.empty_like(weights)
    ops.route_grouped(h.to(DEV), w.to(DEV), correction.to(DEV), top, groups, kept, ids2, weights2)
    device_score = torch.empty(rows, experts, device=DEV)        # the kernel's own float32 scores: sums of them decide between groups
    every = torch.empty(rows, experts, dtype=torch.int32, device=DEV)
    ops.route_topk(h.to(DEV), w.to(DEV), experts, every, device_score)
    plain = torch.empty(rows, experts)
    plain.scatter_(1, every.cpu().long(), device_score.cpu())
    for r in range(rows):
        choice, per = plain[r] + correction, experts // groups
        if groups > 1:
            two = choice.view(groups, per).topk(min(2, per), dim=1).values
            keep = picks((two.sum(1) if per > 1 else two[:, 0]).tolist(), kept)
            choice = torch.where(torch.isin(torch.arange(experts) // per, torch.tensor(keep)), choice, torch.tensor(-float("inf")))
        assert ids2[r].cpu().tolist() == picks(choice.tolist(), top)
        if nan and r == rows - 1:
            assert weights2[r].isnan().all()
            continue
        # float32 sums of up to 64 scores: 63 roundings of at most the sum, one of the quotient, one of the product
        picked = plain[r][ids2[r].cpu().long()].double()
        torch.testing.assert_close(weights2[r].double().cpu(), picked / picked.sum(), rtol=65 * 2.0 ** -24, atol=0.0)


@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5, 16])
@pytest.mark.parametrize("H,G,d,dv,rope,pairing", [(2, 1, 128, 128, 128, 0), (3, 1, 136, 64, 64, 1), (1, 1, 512, 512, 16, 0), (2, 2, 8, 130, 0, 0)])
@pytest.mark.parametrize("dtype", [F32, BF16])
def test_convolved_heads_of_single_rows(ops, H, G, d, dv, rope, pairing, taps, dtype):
    """Four taps on 16 bytes are one load, up to four others a load each, more go the form for portions; heads of up to 128 lanes and wider
    ones have instances of their own."""
    g = torch.Generator().manual_seed(d + taps)
    rows, page, channels = 5, 16, H * d + G * (d + dv)
    joint = torch.randn(rows, channels, generator=g).to(dtype).to(DEV)
    conv, bias = torch.randn(channels, taps, generator=g).to(DEV), torch.randn(channels, generator=g).to(DEV)
    state = torch.randn(7, taps - 1, channels, generator=g).to(dtype).to(DEV)
    qw, kw = torch.rand(d, generator=g).to(DEV), torch.rand(d, generator=g).to(DEV)
    cos, sin = (torch.rand(64, max(rope // 2, 1), generator=g)[:, :rope // 2].contiguous().to(DEV) for _ in range(2))
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)
    row_pos, row_seg, slots = i32(0, 2, 17, 40, 9), i32(0, 1, 2, 3, -1), i32(6, 0, 3, 1, 0)
    tables, seg_start = torch.arange(20, dtype=torch.int32, device=DEV).view(5, 4), torch.arange(6, dtype=torch.int32, device=DEV)
    results = []
    for form, single in ((lambda t: t, True), (off, True), (lambda t: t, False)):
        st, q = state.clone(), torch.zeros(rows, H * d, dtype=dtype, device=DEV)
        k, v = torch.zeros(20, G, d // 8, page, 8, dtype=dtype, device=DEV), torch.zeros(20, G, dv, page, dtype=dtype, device=DEV)
        ops.conv_qkv_store(joint, form(conv), bias, st, qw, kw, 1e-5, q, row_pos, row_seg, seg_start, slots, tables, cos, sin, k, v, H, G, d, dv, rope,
                           pairing, page, 8, single_rows=single)
        results.append((q, k, v, st))
    for other in results[1:]:
        for a, b in zip(results[0], other):
            assert torch.equal(a, b)
    assert not results[0][0][4].any() and torch.equal(results[0][3][[2, 4, 5]], state[[2, 4, 5]])


@pytest.mark.parametrize("width", [4, 1020, 1536, 2048, 2052])
@pytest.mark.parametrize("dtype", [F32, BF16])
def test_norms_with_four_taps(ops, width, dtype):
    g = torch.Generator().manual_seed(width)
    rows = 3
    x, w1, w2 = torch.randn(rows, width, generator=g).to(DEV), torch.rand(width, generator=g).to(DEV), torch.rand(width, generator=g).to(DEV)
    conv, state = torch.randn(width, 4, generator=g).to(DEV), torch.randn(4, 3, width, generator=g).to(dtype).to(DEV)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)
    row_seg, slots = i32(0, 1, -1), i32(3, 1, 0)
    results = []
    for taps in (conv, off(conv)):
        a, b = state.clone(), state.clone()
        outs = [torch.full((rows, width), 7.0, dtype=dtype, device=DEV) for _ in range(3)]
        ops.norm_short_conv(x, w1, 1e-5, taps, a, row_seg, slots, outs[0])
        assert ops.layernorm_conv(x, w1, 1e-5, taps, b, row_seg, slots, outs[1], w2, 1e-3, outs[2])
        results.append(outs + [a, b])
    for a, b in zip(*results):
        assert torch.equal(a, b)
    assert not any(o[2].any() for o in results[0][:3]) and all(torch.equal(s[[0, 2]], state[[0, 2]]) for s in results[0][3:])


@pytest.mark.parametrize("width,taps", [(40, 1), (40, 3), (1020, 4), (2048, 2), (2052, 3), (2052, 4), (5000, 1)])
@pytest.mark.parametrize("dtype", [F32, BF16])
def test_norms_with_few_taps_and_with_more(ops, width, taps, dtype):
    """Up to four taps and more of them are kernels of their own, rows of up to 2,048 lanes and wider ones instances: taps of zero ahead of the
    others leave the bits as they are, whatever the entries that they meet."""
    g = torch.Generator().manual_seed(width + taps)
    rows, ahead = 3, 6 - taps
    x, w1, w2 = torch.randn(rows, width, generator=g).to(DEV), torch.rand(width, generator=g).to(DEV), torch.rand(width, generator=g).to(DEV)
    conv, state = torch.randn(width, taps, generator=g).to(DEV), torch.randn(4, taps - 1, width, generator=g).to(dtype).to(DEV)
    conv6, state6 = torch.cat([torch.zeros(width, ahead, device=DEV), conv], 1), torch.cat([torch.randn(4, ahead, width, generator=g).to(dtype).to(DEV), state], 1)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)
    row_seg, slots = i32(0, 1, -1), i32(3, 1, 0)
    results = []
    for w, st in ((conv, state), (conv6, state6)):
        a, b = st.clone(), st.clone()
        outs = [torch.full((rows, width), 7.0, dtype=dtype, device=DEV) for _ in range(4)]
        ops.norm_short_conv(x, w1, 1e-5, w, a if w.shape[1] > 1 else None, row_seg, slots, outs[0])
        assert ops.layernorm_conv(x, w1, 1e-5, w, b if w.shape[1] > 1 else None, row_seg, slots, outs[1], w2, 1e-3, outs[2])
        assert ops.layernorm_conv(x, w1, 1e-5, w, st.clone() if w.shape[1] > 1 else None, row_seg, slots, outs[3])      # one norm
        results.append(outs + [t[:, t.shape[1] - (taps - 1):] for t in (a, b)])
    for one, other in zip(*results):
        assert torch.equal(one, other)
    assert torch.equal(results[0][1], results[0][3]) and not any(o[2].any() for o in results[0][:4])
    assert all(torch.equal(t[[0, 2]], state[[0, 2]]) for t in results[0][4:])


@pytest.mark.parametrize("width", [4, 1024, 1028, 2044, 4096, 8192])
@pytest.mark.parametrize("branch", [F32, BF16])
@pytest.mark.parametrize("out", [F32, BF16])
def test_sums_and_norms_off_16_bytes(ops, width, branch, out):
    """Branch and output on 16 bytes go four values at a time, others one by one."""
    g = torch.Generator().manual_seed(width)
    x, w = torch.randn(3, width, generator=g).to(DEV), torch.rand(width, generator=g).to(DEV)
    add = torch.randn(3, width, generator=g).to(branch).to(DEV)
    results = []
    for form in (lambda t: t, off):
        y, to = x.clone(), form(torch.zeros(3, width, dtype=out, device=DEV))
        ops.add_rmsnorm(y, form(add), w, 1e-5, to)
        results.append((y, to))
    assert torch.equal(results[0][0], x + add.float()) and torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


@pytest.mark.parametrize("H,G,d,dv,rope", [(4, 2, 64, 64, 64), (3, 1, 40, 24, 16), (8, 8, 128, 128, 0), (32, 8, 128, 128, 128), (26, 2, 128, 64, 64), (33, 1, 96, 32, 0)])
@pytest.mark.parametrize("start", [0, 8, 3])
def test_rotated_portions_in_pieces_of_a_thread(ops, H, G, d, dv, rope, start):
    """256 rows and more go eight rows a workgroup, from more than 3,072 pieces of eight lanes in eight rows on (the last three sizes: 5,120, 3,584 and
    3,264) four pieces of a thread together, fewer rows a row a workgroup: rows in runs of eight tokens of one request, runs that a request's end
    cuts, a ragged last group, whose threads have fewer pieces than four or none, and padding rows."""
    g = torch.Generator().manual_seed(d + start)
    counts, page = [(0, 131), (1, 77), (2, 68)], 16
    pos = torch.cat([torch.arange(start, start + n) for _, n in counts] + [torch.zeros(5, dtype=torch.int64)]).int().to(DEV)
    seg = torch.cat([torch.full((n,), s) for s, n in counts] + [torch.full((5,), -1)]).int().to(DEV)
    rows = pos.numel()
    tables = torch.randperm(36, generator=g).int().view(3, 12).to(DEV)
    qkv = torch.randn(rows, (H + G) * d + G * dv, generator=g).to(BF16).to(DEV)
    cos, sin = (torch.rand(192, max(rope // 2, 4), generator=g).to(DEV) for _ in range(2))
    cos, sin = (t[:, :rope // 2].contiguous() for t in (cos, sin))
    results = []
    for step in (rows, 100):
        x = qkv.clone()
        k, v = torch.zeros(36, G, d // 8, page, 8, dtype=BF16, device=DEV), torch.zeros(36, G, dv, page, dtype=BF16, device=DEV)
        for a in range(0, rows, step):
            part = x[a:a + step]
            ops.rope_kv_store(part, pos[a:a + step].contiguous(), seg[a:a + step].contiguous(), tables, cos, sin, k, v, H, G, d, rope, 1, page, v_dim=dv)
        results.append((x, k, v))
    for a, b in zip(*results):
        assert torch.equal(a, b)
