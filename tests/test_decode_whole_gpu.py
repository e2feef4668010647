"""Decode attention over contexts that one workgroup takes whole (heads of 128 lanes, 512 keys at most): around the end of its first round of 256
keys and of its second, and where a bound of 513 splits them again.  Reference and tolerance of test_decode_attention_edges_gpu.py."""
import pytest
import torch
from test_decode_attention_edges_gpu import reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads", [(12, 2), (4, 4), (20, 1)])
@pytest.mark.parametrize("ps", [8, 16, 64])
@pytest.mark.parametrize("bound,contexts", [(512, [1, 64, 255, 256, 257, 320, 511, 512]), (513, [256, 257, 513])])
def test_whole_contexts(bound, contexts, heads, kv_heads, ps):
    from fllm_amd.kernels import Ops
    ops, d, rows = Ops(), 128, len(contexts)
    gen = torch.Generator().manual_seed(bound + ps)
    per = [-(-n // ps) for n in contexts]
    order = torch.randperm(sum(per), generator=gen) + 1                    # page 0 belongs to nobody
    kp = torch.full((sum(per) + 1, kv_heads, d // 8, ps, 8), float("nan"), dtype=torch.bfloat16)
    vp = torch.full((sum(per) + 1, kv_heads, d, ps), float("nan"), dtype=torch.bfloat16)
    tables = torch.zeros((rows, max(per)), dtype=torch.int32)
    q = torch.randn((rows, heads * d), generator=gen).to(torch.bfloat16)
    want = torch.empty((rows, heads * d), dtype=torch.float64)
    for r, n in enumerate(contexts):
        mine, order = order[:per[r]], order[per[r]:]
        tables[r, :per[r]] = mine.to(torch.int32)
        k, v = (torch.randn((kv_heads, n, d), generator=gen).to(torch.bfloat16) for _ in range(2))
        for t in range(n):
            kp[mine[t // ps], :, :, t % ps] = k[:, t].view(kv_heads, d // 8, 8)
            vp[mine[t // ps], :, :, t % ps] = v[:, t]
        want[r] = reference(q[r].view(heads, d).double(), k.double(), v.double(), n, 0, kv_heads, d ** -0.5, None).flatten()
    out = torch.empty((rows, heads * d), dtype=torch.bfloat16, device="cuda")
    space = torch.empty(ops.attention_workspace_bytes(rows, heads, kv_heads, d, bound) + 16, dtype=torch.uint8, device="cuda")
    seg, start = (torch.arange(n, dtype=torch.int32, device="cuda") for n in (rows, rows + 1))
    ops.attention(q.cuda(), kp.cuda(), vp.cuda(), tables.cuda(), torch.tensor(contexts, dtype=torch.int32, device="cuda") - 1, seg, start, out, heads, kv_heads,
                  d, ps, d ** -0.5, None, bound, uniform_rows=1, workspace=space)
    got = out.double().cpu()
    assert torch.isfinite(got).all() and (got - want).abs().max() <= 2 ** -7 * want.abs().max()
