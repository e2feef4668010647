"""Row kernels whose rows are shared among workgroups, at the edges of a workgroup's piece: every value is written, none beyond."""
import pytest
import torch

from reference_ops import ReferenceOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LOUD = 1e4


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


# values of a row: 4, 1,023 and 1,025 beside a workgroup's 1,024, several pieces, and lanes beyond the rotated ones
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,heads,dim,vdim,rope", [(1, 1, 1, 2, 0), (3, 1, 340, 343, 6), (2, 1, 340, 344, 340), (5, 1, 341, 343, 2), (2, 12, 128, 128, 128),
                                                      (1, 16, 128, 256, 64), (70, 2, 64, 64, 32)])
def test_rotated_operands_in_pieces(ops, rows, heads, dim, vdim, rope, dtype):
    g = torch.Generator().manual_seed(dim)
    width = heads * (2 * dim + vdim)
    qkv = torch.randn(rows, width + 3, generator=g).to(dtype)
    pos = torch.randint(0, 50, (rows,), generator=g, dtype=torch.int32)
    cos, sin = torch.rand(50, rope // 2, generator=g) * 2 - 1, torch.rand(50, rope // 2, generator=g) * 2 - 1
    want = torch.empty(rows, width, dtype=torch.float64)
    ReferenceOps().rotate_scale(qkv.double(), want, pos, cos, sin, heads, dim, vdim, rope, 0.3)
    room = torch.full((rows + 1, width), LOUD, device=DEV)
    ops.rotate_scale(qkv.to(DEV), room[:rows], pos.to(DEV), cos.to(DEV), sin.to(DEV), heads, dim, vdim, rope, 0.3)
    got = room[:rows].double().cpu()
    # two products and a sum of numbers below 5 in float32, times the key's factor
    assert ((got - want).abs() <= 4 * 2.0 ** -24 * (want.abs() + 5)).all()
    assert (room[rows] == LOUD).all()


# head sizes on both sides of what a wave holds at once (256 lanes); heads that fill workgroups, leave one wave, or are fewer than its waves
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,H,G,d,dv", [(1, 1, 1, 8, 8), (4, 12, 2, 128, 128), (3, 3, 2, 64, 24), (5, 2, 1, 256, 40), (2, 3, 1, 257, 16), (2, 2, 2, 320, 300),
                                           (3, 1, 1, 20, 700), (513, 3, 2, 40, 16)])
def test_heads_normed_and_stored_a_head_a_wave(ops, rows, H, G, d, dv, dtype):
    g = torch.Generator().manual_seed(d + H)
    page, chunk = 16, 8 if d % 8 == 0 else 1
    qkv = torch.randn(rows, (H + G) * d + G * dv, generator=g).to(dtype)
    pos = torch.randint(0, 3 * page, (rows,), generator=g, dtype=torch.int32)
    seg = torch.arange(rows, dtype=torch.int32)
    if rows > 2:
        seg[1] = -1                                    # a padding row
    tables = torch.randperm(3 * rows + 2, generator=g)[:3 * rows].to(torch.int32).view(rows, 3).contiguous()
    k = torch.full((3 * rows + 2, G, d // chunk, page, chunk), LOUD).to(dtype)
    v = torch.full((3 * rows + 2, G, dv, page), LOUD).to(dtype)
    for store in (True, False):
        want = [t.clone() for t in (qkv, k, v)]
        got = [t.to(DEV) for t in (qkv, k, v)]
        ReferenceOps().head_norm_kv_store(want[0], 1e-5, d, pos, seg, tables, want[1] if store else None, want[2] if store else None, H, G, d, page,
                                          v_dim=dv, key_chunk=chunk)
        ops.head_norm_kv_store(got[0], 1e-5, d, pos.to(DEV), seg.to(DEV), tables.to(DEV), got[1] if store else None, got[2] if store else None,
                               H, G, d, page, v_dim=dv, key_chunk=chunk)
        eps = 2.0 ** -7 if dtype == torch.bfloat16 else 1e-6 * (d / 64 + 1)      # one rounding to the row's type; a float32 sum
        for name, a, b in zip(("rows", "keys", "values"), got, want):
            a, b = a.double().cpu(), b.double()
            assert ((a - b).abs() <= eps * b.abs() + 1e-7).all(), name
