"""The forms of the row kernels that read everything a row needs in one round of loads (bfloat16, pieces of 4 and 8 lanes), against the
plain forms of the same entry points, which an operand that begins off a 16-byte boundary selects, and against float64: widths of one piece, of
a whole round of the workgroup and one more, heads whose threads fill no power of two, every norm, rotations of part of a head, padding rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16_EPS = 2.0 ** -8


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


def off(t):
    """A dense copy of t that begins one element behind a 16-byte boundary."""
    out = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    return out.copy_(t)


def alike(got, want, steps=2):
    """Sums in another order, then one rounding.  float32: steps of the largest value, since terms of its size may cancel in a smaller
    one; bfloat16 results of such sums: steps of the value itself, the float32 part of the bound being 2^-14 of it."""
    eps, floor = (BF16_EPS, 1e-2) if got.dtype == torch.bfloat16 else (2.0 ** -23, 1.0)
    want, got = want.float(), got.float()
    assert ((got - want).abs() <= steps * eps * (want.abs() + floor * want.abs().max())).all(), (got - want).abs().max()


@pytest.mark.parametrize("rows,width,experts,top,score", [(1, 8, 8, 2, "sigmoid"), (5, 1536, 8, 2, "softmax"), (3, 2056, 70, 5, "sigmoid"), (2, 512, 3, 3, "softmax")])
def test_routers(ops, rows, width, experts, top, score):
    g = torch.Generator().manual_seed(width)
    h = torch.randn(rows, width, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(experts, width, generator=g) * width ** -0.5 * 2).to(torch.bfloat16).to(DEV)
    correction = torch.rand(experts, generator=g).to(DEV)
    got = [(torch.empty(rows, top, dtype=torch.int32, device=DEV), torch.empty(rows, top, device=DEV)) for _ in range(4)]
    ops.route_topk(h, w, top, *got[0], score=score, renormalize=True, route_scale=2.5)
    ops.route_topk(off(h), w, top, *got[1], score=score, renormalize=True, route_scale=2.5)
    groups = 2 if experts % 2 == 0 else 1
    ops.route_grouped(h, w, correction, top, groups, groups, *got[2], route_scale=2.5)
    ops.route_grouped(off(h), w, correction, top, groups, groups, *got[3], route_scale=2.5)
    for a, b in ((got[0], got[1]), (got[2], got[3])):
        assert torch.equal(a[0], b[0])
        torch.testing.assert_close(a[1], b[1], rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("parts", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("rows,width", [(3, 4), (2, 1024), (1, 1028), (5, 1536), (2, 4096), (2, 4100)])
@pytest.mark.parametrize("weighted,normed,nexts", [(True, True, torch.bfloat16), (False, False, torch.float32), (True, False, None)])
def test_sums_of_normed_branches(ops, rows, width, parts, weighted, normed, nexts):
    g = torch.Generator().manual_seed(parts * 7 + width)
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV)
    x, branch, gain, pw, nw = rnd(rows, width), rnd(rows * parts, width), rnd(width), rnd(rows, parts), rnd(width)
    outs = []
    for form in (lambda t: t, off):
        y = x.clone()
        nxt = None if nexts is None else torch.empty(rows, width, dtype=nexts, device=DEV)
        ops.postnorm_add(y, form(branch), gain, 1e-5 if normed else None, parts=parts, part_weights=pw if weighted else None,
                         next_weight=None if nexts is None else nw, next_eps=1e-6, next_out=nxt)
        outs.append((y, nxt))
    alike(outs[0][0], outs[1][0], 8)
    if nexts is not None:
        alike(outs[0][1], outs[1][1], 8 if nexts == torch.float32 else 2)


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("heads,kv_heads,k_dim,v_dim,rope,keys_are_values,store", [
    (12, 2, 128, 128, 128, False, True), (3, 1, 24, 40, 16, False, True), (5, 5, 512, 512, 256, True, True), (20, 4, 64, 32, 0, False, True),
    (40, 8, 64, 64, 32, False, False)])
def test_normed_and_rotated_heads(ops, mode, heads, kv_heads, k_dim, v_dim, rope, keys_are_values, store):
    g = torch.Generator().manual_seed(heads * k_dim + mode)
    rows, page, pages = 5, 16, 4
    wide = heads * k_dim + kv_heads * (k_dim + (0 if keys_are_values else v_dim))
    qkv = torch.randn(rows, wide + 8, generator=g).to(torch.bfloat16).to(DEV)
    qw, kw = (1.0 + 0.1 * torch.randn(n * k_dim if mode == 2 else k_dim, generator=g) for n in (heads, kv_heads))
    angles = torch.rand(64, rope // 2, generator=g) * 6.0
    cos, sin = torch.cos(angles).contiguous().to(DEV), torch.sin(angles).contiguous().to(DEV)
    pos = torch.tensor([0, 15, 16, 37, 5], dtype=torch.int32, device=DEV)
    seg = torch.tensor([0, 0, 1, 1, -1], dtype=torch.int32, device=DEV)
    tables = torch.tensor([[3, 1, 0], [2, 0, 1]], dtype=torch.int32, device=DEV)
    blend = None if keys_are_values else torch.randn(rows, kv_heads * v_dim, generator=g).to(torch.bfloat16).to(DEV)
    amount = torch.tensor([0.3], device=DEV)
    outs = []
    for form in (lambda t: t, off):
        q = torch.zeros(rows, heads * k_dim, dtype=torch.bfloat16, device=DEV)
        k = torch.zeros(pages, kv_heads, k_dim // 8, page, 8, dtype=torch.bfloat16, device=DEV)
        v = torch.zeros(pages, kv_heads, v_dim, page, dtype=torch.bfloat16, device=DEV)
        ops.normed_rope_store(form(qkv), mode, qw.to(DEV) if mode else None, kw.to(DEV) if mode else None, 1e-5, q, pos, seg, tables, cos, sin,
                              k if store else None, v if store else None, heads, kv_heads, k_dim, v_dim, rope,
                              page, 8, values_from_keys=keys_are_values, blend=blend, blend_amount=amount if blend is not None else None)
        outs.append((q[:4], k, v))
    for a, b in zip(*outs):
        alike(a, b)
    assert torch.equal(outs[0][2], outs[1][2])          # values are stored, or blended in float32, alike


@pytest.mark.parametrize("form", ["heads", "projections"])
def test_keys_that_begin_off_16_bytes_are_stored_by_the_plain_form(ops, form):
    """Pieces of 16 bytes go to pages that begin on 16 bytes only: the same bits as the plain form, which operands off that boundary select."""
    g = torch.Generator().manual_seed(3)
    rows, page, pages, heads, kv_heads, dim = 5, 16, 4, 12, 2, 128
    qkv = torch.randn(rows, (heads + 2 * kv_heads) * dim, generator=g).to(torch.bfloat16).to(DEV)
    qw, kw = (1.0 + 0.1 * torch.randn(dim if form == "heads" else n * dim, generator=g).to(DEV) for n in (heads, kv_heads))
    angles = torch.rand(64, dim // 2, generator=g) * 6.0
    cos, sin = torch.cos(angles).contiguous().to(DEV), torch.sin(angles).contiguous().to(DEV)
    pos = torch.tensor([0, 15, 16, 37, 5], dtype=torch.int32, device=DEV)
    seg = torch.tensor([0, 0, 1, 1, -1], dtype=torch.int32, device=DEV)
    tables = torch.tensor([[3, 1, 0], [2, 0, 1]], dtype=torch.int32, device=DEV)
    outs = []
    for rows_as, pages_as in ((off, lambda t: t), (lambda t: t, off)):
        q = torch.zeros(rows, heads * dim, dtype=torch.bfloat16, device=DEV)
        k = pages_as(torch.zeros(pages, kv_heads, dim // 8, page, 8, dtype=torch.bfloat16, device=DEV))
        v = torch.zeros(pages, kv_heads, dim, page, dtype=torch.bfloat16, device=DEV)
        if form == "heads":
            ops.normed_rope_store(rows_as(qkv), 1, qw, kw, 1e-5, q, pos, seg, tables, cos, sin, k, v, heads, kv_heads, dim, dim, dim, page, 8)
        else:
            ops.qk_norm_rope_store(rows_as(qkv), qw, kw, 1e-5, q, pos, seg, tables, cos, sin, k, v, heads, kv_heads, dim, dim, dim, page, 8)
        outs.append((q[:4], k, v))
    assert all(torch.equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("x_type", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,weighted", [(1, 4, True), (3, 1536, True), (2, 2052, False), (2, 8192, True)])
def test_gated_norms(ops, rows, width, weighted, x_type):
    g = torch.Generator().manual_seed(width)
    x = torch.randn(rows, width, generator=g).to(x_type).to(DEV)
    gate = torch.randn(rows, width + 12, generator=g).to(torch.bfloat16).to(DEV)[:, 12:]
    w = torch.randn(width, generator=g).to(DEV) if weighted else None
    outs = [torch.empty(rows, width, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    ops.gated_norm(x, w, 1e-5, gate, outs[0])
    ops.gated_norm(off(x), w, 1e-5, gate, outs[1])
    alike(*outs)


@pytest.mark.parametrize("rows,width", [(1, 8), (3, 8960), (2, 16392), (1, 32768)])
def test_polynomial_activation(ops, rows, width):
    z = torch.randn(rows, width, generator=torch.Generator().manual_seed(width)).to(torch.bfloat16).to(DEV)
    coeffs = torch.tensor([0.7, -0.4, 0.2, 0.1], device=DEV)
    outs = [torch.empty_like(z) for _ in range(2)]
    ops.polynorm(z, coeffs, 1e-5, outs[0])
    ops.polynorm(off(z), coeffs, 1e-5, outs[1])
    alike(*outs)


@pytest.mark.parametrize("vocab", [5, 8192, 8193, 50000])
def test_adjusted_logits_over_spans(ops, vocab):
    """Rows of several spans: penalties, biases, blocked ids and allow lists at the spans' edges, against the plain functions."""
    from fllm_amd.sampling import SamplingParams
    from fllm_amd.sampling.adjust import AdjustRow, pack
    from reference_ops import ReferenceOps
    edge = sorted({t for t in (0, 4, 8191, 8192, vocab - 1) if t < vocab})
    rows = [AdjustRow(SamplingParams(repetition_penalty=1.3, presence_penalty=0.2, frequency_penalty=0.1, logit_bias=tuple((t, 0.5) for t in edge)),
                      {t: 2 for t in edge}, blocked=(edge[-1], vocab + 3), last_row=0),
            None,
            AdjustRow(SamplingParams(allowed_token_ids=tuple(edge)), {}, allowed=tuple(edge)),
            AdjustRow(SamplingParams(allowed_token_ids=(1, 2, vocab + 9)), {}, allowed=(1, 2, vocab + 9), pairs=((edge[0], 2),), last_row=1)]
    packed, sections = pack(rows)
    logits = torch.randn(len(rows), vocab, generator=torch.Generator().manual_seed(vocab))
    last = torch.tensor([edge[-1], edge[0]], dtype=torch.int32)
    want = ReferenceOps().adjust_logits(logits.clone(), packed, sections, last)
    got = ops.adjust_logits(logits.clone().to(DEV), packed.to(DEV), sections, last.to(DEV)).cpu()
    torch.testing.assert_close(got, want.float(), rtol=1e-6, atol=1e-6)


def test_allow_lists_that_do_not_rise_stay_inside_their_row(ops):
    """The lists are the caller's word to rise; one that does not may block more than it says, and nothing outside of its row."""
    from fllm_amd.sampling import SamplingParams
    from fllm_amd.sampling.adjust import AdjustRow, pack
    vocab, listed = 20000, (3, 700, 8191, 8192, 12000, 19999)
    packed, sections = pack([None, AdjustRow(SamplingParams(allowed_token_ids=listed), {}, allowed=listed), None])
    words = packed.tolist()
    at = next(i for i in range(len(words)) if tuple(words[i:i + len(listed)]) == listed)
    logits = torch.randn(3, vocab, generator=torch.Generator().manual_seed(1))
    blocked = [t for t in range(vocab) if t not in listed]
    for order in ((19999, 12000, 8192, 8191, 700, 3), (8192, 3, 19999, 700, 12000, 8191), (12000, 19999, 3, 8191, 8192, 700)):
        packed[at:at + len(listed)] = torch.tensor(order, dtype=torch.int32)
        got = ops.adjust_logits(logits.clone().to(DEV), packed.to(DEV), sections).cpu()
        assert torch.equal(got[0], logits[0]) and torch.equal(got[2], logits[2])
        assert (got[1, blocked] == float("-inf")).all()
        assert all(got[1, t] in (logits[1, t], float("-inf")) for t in listed)


def near(got, exact):
    """Against float64: one rounding to bfloat16 (at most 2^-8 of the value; a float32 result has none that counts) behind sums of up to 32,768
    float32 terms, whose errors stay below 2^-18 of the largest value."""
    eps = 2.0 ** -8 if got.dtype == torch.bfloat16 else 0.0
    got, exact = got.double().cpu(), exact.double()
    assert ((got - exact).abs() <= eps * exact.abs() + 2.0 ** -18 * exact.abs().max()).all(), ((got - exact).abs() / exact.abs().max()).max()


@pytest.mark.parametrize("rows,width,experts,top,score", [(1, 8, 8, 2, "sigmoid"), (5, 1536, 8, 2, "softmax"), (3, 2056, 70, 5, "sigmoid"), (2, 512, 3, 3, "softmax")])
def test_routers_against_float64(ops, rows, width, experts, top, score):
    from reference_ops import ReferenceOps
    g = torch.Generator().manual_seed(width + 1)
    h = torch.randn(rows, width, generator=g).to(torch.bfloat16)
    w = (torch.randn(experts, width, generator=g) * width ** -0.5 * 2).to(torch.bfloat16)
    correction = torch.rand(experts, generator=g)
    groups = 2 if experts % 2 == 0 else 1
    new = lambda d: (torch.empty(rows, top, dtype=torch.int32, device=d), torch.empty(rows, top, device=d))
    for call in (lambda o, d, out: o.route_topk(h.to(d), w.to(d), top, *out, score=score, renormalize=True, route_scale=2.5),
                 lambda o, d, out: o.route_grouped(h.to(d), w.to(d), correction.to(d), top, groups, groups, *out, route_scale=2.5)):
        got, want = new(DEV), new("cpu")
        call(ops, DEV, got)
        call(ReferenceOps(), "cpu", want)
        assert torch.equal(got[0].cpu(), want[0])
        torch.testing.assert_close(got[1].cpu(), want[1], rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("parts", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("rows,width", [(3, 4), (2, 1024), (1, 1028), (5, 1536), (2, 4096), (2, 4100)])
@pytest.mark.parametrize("weighted,normed,nexts", [(True, True, torch.bfloat16), (False, False, torch.float32), (True, False, None)])
def test_sums_of_normed_branches_against_float64(ops, rows, width, parts, weighted, normed, nexts):
    from reference_ops import ReferenceOps
    g = torch.Generator().manual_seed(parts * 11 + width)
    x, branch, gain, pw, nw = (torch.randn(*s, generator=g) for s in ((rows, width), (rows * parts, width), (width,), (rows, parts), (width,)))
    results = []
    for o, d, of in ((ops, DEV, lambda t: t), (ReferenceOps(), "cpu", lambda t: t.double())):
        y = of(x.to(d, copy=True))
        nxt = None if nexts is None else torch.empty(rows, width, dtype=nexts if d == DEV else torch.float64, device=d)
        o.postnorm_add(y, of(branch.to(d)), of(gain.to(d)), 1e-5 if normed else None, parts=parts, part_weights=of(pw.to(d)) if weighted else None,
                       next_weight=None if nexts is None else of(nw.to(d)), next_eps=1e-6, next_out=nxt)
        results.append((y, nxt))
    near(results[0][0], results[1][0])
    if nexts is not None:
        near(results[0][1], results[1][1])


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("heads,kv_heads,k_dim,v_dim,rope,keys_are_values", [(12, 2, 128, 128, 128, False), (3, 1, 24, 40, 16, False), (5, 5, 512, 512, 256, True),
                                                                             (20, 4, 64, 32, 0, False)])
def test_normed_and_rotated_heads_against_float64(ops, mode, heads, kv_heads, k_dim, v_dim, rope, keys_are_values):
    from reference_ops import ReferenceOps
    g = torch.Generator().manual_seed(heads * k_dim + mode + 1)
    rows, page, pages = 5, 16, 4
    wide = heads * k_dim + kv_heads * (k_dim + (0 if keys_are_values else v_dim))
    qkv = torch.randn(rows, wide + 8, generator=g).to(torch.bfloat16)
    qw, kw = (1.0 + 0.1 * torch.randn(n * k_dim if mode == 2 else k_dim, generator=g) for n in (heads, kv_heads))
    angles = torch.rand(64, rope // 2, generator=g) * 6.0
    cos, sin = torch.cos(angles).contiguous(), torch.sin(angles).contiguous()
    pos, seg = torch.tensor([0, 15, 16, 37, 5], dtype=torch.int32), torch.tensor([0, 0, 1, 1, -1], dtype=torch.int32)
    tables = torch.tensor([[3, 1, 0], [2, 0, 1]], dtype=torch.int32)
    blend = None if keys_are_values else torch.randn(rows, kv_heads * v_dim, generator=g).to(torch.bfloat16)
    amount = torch.tensor([0.3])
    results = []
    for o, d, kind in ((ops, DEV, torch.bfloat16), (ReferenceOps(), "cpu", torch.float64)):
        at = lambda t: None if t is None else t.to(d)
        q = torch.zeros(rows, heads * k_dim, dtype=kind, device=d)
        k = torch.zeros(pages, kv_heads, k_dim // 8, page, 8, dtype=kind, device=d)
        v = torch.zeros(pages, kv_heads, v_dim, page, dtype=kind, device=d)
        o.normed_rope_store(at(qkv if d == DEV else qkv.double()), mode, at(qw) if mode else None, at(kw) if mode else None, 1e-5, q, at(pos), at(seg), at(tables),
                            at(cos), at(sin), k, v, heads, kv_heads, k_dim, v_dim, rope, page, 8, values_from_keys=keys_are_values,
                            blend=at(blend), blend_amount=at(amount) if blend is not None else None)
        results.append((q[:4], k, v))
    for a, b in zip(*results):
        near(a, b)


@pytest.mark.parametrize("x_type", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,weighted", [(1, 4, True), (3, 1536, True), (2, 2052, False), (2, 8192, True)])
def test_gated_norms_against_float64(ops, rows, width, weighted, x_type):
    from reference_ops import ReferenceOps
    g = torch.Generator().manual_seed(width + 1)
    x, w = torch.randn(rows, width, generator=g).to(x_type), torch.randn(width, generator=g) if weighted else None
    gate = torch.randn(rows, width + 12, generator=g).to(torch.bfloat16)[:, 12:]
    got, want = torch.empty(rows, width, dtype=torch.bfloat16, device=DEV), torch.empty(rows, width, dtype=torch.float64)
    wide = torch.zeros(rows, width + 12, dtype=torch.bfloat16, device=DEV)
    wide[:, 12:] = gate.to(DEV)
    ops.gated_norm(x.to(DEV), w.to(DEV) if weighted else None, 1e-5, wide[:, 12:], got)
    ReferenceOps().gated_norm(x, w, 1e-5, gate, want)
    near(got, want)


@pytest.mark.parametrize("rows,width", [(1, 8), (3, 8960), (2, 16392), (1, 32768)])
def test_polynomial_activation_against_float64(ops, rows, width):
    from reference_ops import ReferenceOps
    z = torch.randn(rows, width, generator=torch.Generator().manual_seed(width + 1)).to(torch.bfloat16)
    coeffs = torch.tensor([0.7, -0.4, 0.2, 0.1])
    got, want = torch.empty(rows, width, dtype=torch.bfloat16, device=DEV), torch.empty(rows, width, dtype=torch.float64)
    ops.polynorm(z.to(DEV), coeffs.to(DEV), 1e-5, got)
    ReferenceOps().polynorm(z, coeffs, 1e-5, want)
    near(got, want)
