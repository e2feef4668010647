"""Decode attention where its blocks end: contexts around 32 and 64 keys, a workgroup's round and the parts of a split, page
sizes below and above a block, windows and chunks that start inside one, more query heads than a tile, a workspace that
is only 4-byte aligned, and slots without a token that hold NaNs.  Against float64 on the CPU.  Tolerance: the probabilities
and the result are rounded to bfloat16 (2^-9 each) beside sums that stay in float32: 2^-7 of the largest value."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CONTEXTS = [1, 31, 32, 33, 63, 64, 65, 127, 255, 256, 257, 511, 513, 1000]


def reference(q, keys, values, n, lo, kv_heads, scale, sinks):
    heads, d = q.shape
    out = torch.empty((heads, d), dtype=torch.float64)
    for h in range(heads):
        k, v = keys[h * kv_heads // heads, lo:n], values[h * kv_heads // heads, lo:n]
        z = (k @ q[h]) * scale
        top = z.max() if sinks is None else max(z.max(), sinks[h])
        e = torch.exp(z - top)
        out[h] = (e @ v) / (e.sum() + (0.0 if sinks is None else torch.exp(sinks[h] - top)))
    return out


@pytest.mark.parametrize("d,heads,kv_heads", [(128, 8, 2), (64, 8, 8), (32, 40, 2)])
@pytest.mark.parametrize("ps", [8, 16, 32, 64])
@pytest.mark.parametrize("window,chunk,sink", [(0, 0, False), (45, 0, True), (0, 70, False)])
def test_decode_attention_at_its_edges(d, heads, kv_heads, ps, window, chunk, sink):
    from fllm_amd.kernels import Ops
    ops = Ops()
    gen = torch.Generator().manual_seed(d + ps + window)
    rows = len(CONTEXTS)
    per = [-(-n // ps) for n in CONTEXTS]
    pages = sum(per) + 1
    order = torch.randperm(pages - 1, generator=gen) + 1                   # page 0 belongs to nobody
    kp = torch.full((pages, kv_heads, d // 8, ps, 8), float("nan"), dtype=torch.bfloat16)
    vp = torch.full((pages, kv_heads, d, ps), float("nan"), dtype=torch.bfloat16)
    tables = torch.zeros((rows, max(per)), dtype=torch.int32)
    q = torch.randn((rows, heads * d), generator=gen).to(torch.bfloat16)
    sinks = torch.randn(heads, generator=gen) if sink else None
    want = torch.empty((rows, heads * d), dtype=torch.float64)
    at = 0
    for r, n in enumerate(CONTEXTS):
        mine = order[at:at + per[r]]
        at += per[r]
        tables[r, :per[r]] = mine.to(torch.int32)
        k = torch.randn((kv_heads, n, d), generator=gen).to(torch.bfloat16)
        v = torch.randn((kv_heads, n, d), generator=gen).to(torch.bfloat16)
        for t in range(n):
            kp[mine[t // ps], :, :, t % ps] = k[:, t].view(kv_heads, d // 8, 8)
            vp[mine[t // ps], :, :, t % ps] = v[:, t]
        lo = max(0, n - window) if window else 0
        if chunk:
            lo = max(lo, (n - 1) // chunk * chunk)
        want[r] = reference(q[r].view(heads, d).double(), k.double(), v.double(), n, lo, kv_heads, d ** -0.5,
                            None if sinks is None else sinks.double()).flatten()
    dev = lambda t: None if t is None else t.cuda()
    most = max(CONTEXTS)
    args = (dev(q), dev(kp), dev(vp), dev(tables), dev(torch.tensor(CONTEXTS, dtype=torch.int32) - 1),
            torch.arange(rows, dtype=torch.int32, device="cuda"), torch.arange(rows + 1, dtype=torch.int32, device="cuda"))
    need = ops.attention_workspace_bytes(rows, heads, kv_heads, d, most)
    results = []
    for offset in (0, 4):
        space = torch.empty(need + 16, dtype=torch.uint8, device="cuda")[offset:offset + max(need, 1)]
        for batch in (rows, 1):               # all rows at once, and the longest context alone (more parts)
            a = list(args)
            if batch == 1:
                a[0], a[3], a[4] = a[0][-1:].contiguous(), a[3][-1:].contiguous(), a[4][-1:].contiguous()
                a[5], a[6] = a[5][:1].contiguous(), a[6][:2].contiguous()
            out = torch.empty((batch, heads * d), dtype=torch.bfloat16, device="cuda")
            one = space if batch == rows else torch.empty(ops.attention_workspace_bytes(1, heads, kv_heads, d, most) + 16, dtype=torch.uint8,
                                                          device="cuda")[offset:]
            ops.attention(*a, out, heads, kv_heads, d, ps, d ** -0.5, window or None, most, uniform_rows=1, workspace=one, chunk=chunk or None,
                          sinks=dev(sinks))
            got, exact = out.double().cpu(), want if batch == rows else want[-1:]
            results.append(got)
            error = (got - exact).abs().max() / exact.abs().max()
            assert error <= 2 ** -7, (offset, batch, float(error))
    assert torch.isfinite(torch.cat(results)).all()


@pytest.mark.parametrize("moved", ["keys", "values"])
def test_pages_that_begin_off_16_bytes_go_to_the_plain_kernel(moved):
    """The matrix-core kernels read 16 bytes of keys and of values at a time; pages that begin elsewhere give the plain kernel's bits."""
    from fllm_amd.kernels import Ops
    ops = Ops()
    gen = torch.Generator().manual_seed(9)
    heads, kv_heads, d, ps, contexts = 8, 2, 64, 16, [1, 40, 100]
    pages, rows = 24, len(contexts)
    rnd = lambda *s: torch.randn(*s, generator=gen).to(torch.bfloat16).cuda()
    q, kp, vp = rnd(rows, heads * d), rnd(pages, kv_heads, d // 8, ps, 8), rnd(pages, kv_heads, d, ps)
    tables = torch.randperm(pages, generator=gen)[:rows * 7].view(rows, 7).to(torch.int32).cuda()
    pos = torch.tensor([n - 1 for n in contexts], dtype=torch.int32, device="cuda")
    seg, start = (torch.arange(n, dtype=torch.int32, device="cuda") for n in (rows, rows + 1))
    off = lambda t: torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)

    def run(k, v):
        out = torch.empty((rows, heads * d), dtype=torch.bfloat16, device="cuda")
        space = torch.empty(ops.attention_workspace_bytes(rows, heads, kv_heads, d, 100) + 16, dtype=torch.uint8, device="cuda")
        ops.attention(q, k, v, tables, pos, seg, start, out, heads, kv_heads, d, ps, d ** -0.5, None, 100, uniform_rows=1, workspace=space)
        return out

    got = run(off(kp) if moved == "keys" else kp, off(vp) if moved == "values" else vp)
    ops.set_fast_kernels(False)
    try:
        want = run(kp, vp)
    finally:
        ops.set_fast_kernels(True)
    assert torch.equal(got, want)
