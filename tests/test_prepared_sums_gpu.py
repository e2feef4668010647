"""The sum that norms a branch into the stream and prepares the norm behind it: the stream's bits are those of the plain sum, the
prepared row is the new row times the norm's weight in bfloat16, and its sum of squares is the new row's."""
import pytest
import torch

from fllm_amd.kernels import KernelError

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


@pytest.mark.parametrize("normed", [True, False])
@pytest.mark.parametrize("rows, width, parts", [(1, 4, 1), (3, 1020, 1), (8, 1536, 1), (16, 1536, 2), (5, 1030, 1), (2, 1031, 3), (7, 4096, 4),
                                                (4, 8192, 1), (3, 8192, 2), (2, 8196, 1), (2, 64, 6)])
def test_the_sum_prepares_the_norm_behind_it(ops, rows, width, parts, normed):
    g = torch.Generator().manual_seed(rows * width + parts)
    x, branch = torch.randn(rows, width, generator=g) * 3, torch.randn(rows * parts, width, generator=g)
    gain, w = torch.rand(width, generator=g) + 0.5, torch.rand(width, generator=g) + 0.5
    eps = 1e-5 if normed else None
    plain = x.to(DEV)
    ops.postnorm_add(plain, branch.to(DEV), gain.to(DEV), eps, parts=parts)
    got = x.to(DEV)
    prepared = ops.postnorm_add_prepare(got, branch.to(DEV), gain.to(DEV), eps, w.to(DEV), parts=parts)
    assert prepared.parts == 1 and prepared.x.shape == (rows, width) and prepared.ssq.shape == (rows,)
    assert torch.equal(got, plain)
    assert torch.equal(prepared.x, (got * w.to(DEV)).to(torch.bfloat16))       # one product and one rounding
    want = (got.double().cpu() ** 2).sum(dim=1)
    # a sum of positive numbers in float32: each at most (squares and additions of a chain) width / 256 + 20 roundings off
    assert ((prepared.ssq.double().cpu() - want).abs() <= want * (width / 256 + 20) * 2.0 ** -24).all()


def test_a_sum_of_squares_needs_the_norm(ops):
    x = torch.ones(2, 64, device=DEV)
    with pytest.raises(KernelError):
        ops.postnorm_add(x, x.clone(), torch.ones(64, device=DEV), 1e-5, next_ssq=torch.empty(2, device=DEV))


def test_the_prepared_product_agrees_with_the_norm_in_the_product(ops):
    """Of 1 to 16 rows of a stream, the gated product behind the prepared norm against float64."""
    g = torch.Generator().manual_seed(5)
    K, inter = 1536, 512
    w = (torch.randn(2 * inter, K, generator=g) * K ** -0.5).to(torch.bfloat16)
    for rows in (1, 8, 9, 16):
        x, branch = torch.randn(rows, K, generator=g), torch.randn(rows, K, generator=g)
        gain, nw = torch.rand(K, generator=g) + 0.5, torch.rand(K, generator=g) + 0.5
        stream = x.to(DEV)
        prepared = ops.postnorm_add_prepare(stream, branch.to(DEV), gain.to(DEV), 1e-5, nw.to(DEV))
        outs = [ops.norm_gate_up_swiglu(stream, nw.to(DEV), 1e-5, w.to(DEV), torch.empty(rows, inter, dtype=torch.bfloat16, device=DEV), **how)
                for how in ({}, dict(prepared=prepared))]
        s = stream.double().cpu()
        n = s / (s.pow(2).mean(1, keepdim=True) + 1e-5).sqrt() * nw.double()
        gate, up = (n @ w.double().t()).split(inter, dim=1)
        want = gate * torch.sigmoid(gate) * up
        errors = [(o.double().cpu() - want).abs().max().item() / want.abs().max().item() for o in outs]
        assert errors[1] <= 2 * errors[0] + 2.0 ** -9, errors        # the same roundings: one of the row, one of the result


@pytest.mark.parametrize("rows", [1, 8, 9, 16])
@pytest.mark.parametrize("heads, kv_heads, K", [(12, 2, 1536), (2, 1, 288), (40, 4, 1568)])
def test_a_copy_changes_no_bit_of_the_rotated_product(ops, rows, heads, kv_heads, K):
    """q, k and v behind a prepared norm of widths that are no multiple of 1,024, with the tile-major copy of their matrix and without:
    matrices of few and of unevenly many tiles, whose rows run in tiles of 8."""
    dim, pages = 128, 4
    g = torch.Generator().manual_seed(K + rows)
    w = (torch.randn((heads + 2 * kv_heads) * dim, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(DEV)
    x, branch = torch.randn(rows, K, generator=g).to(DEV), torch.randn(rows, K, generator=g).to(DEV)
    gain = torch.ones(K, device=DEV)
    prepared = ops.postnorm_add_prepare(x, branch, gain, 1e-5, gain)
    pos = torch.arange(rows, dtype=torch.int32, device=DEV)
    seg = torch.zeros(rows, dtype=torch.int32, device=DEV)
    tables = torch.arange(pages, dtype=torch.int32, device=DEV)[None]
    angles = torch.randn(64, dim // 2, generator=g).to(DEV)
    cos, sin = angles.cos(), angles.sin()

    def product():
        q = torch.empty(rows, heads * dim, dtype=torch.bfloat16, device=DEV)
        k = torch.zeros(pages, kv_heads, dim // 8, 16, 8, dtype=torch.bfloat16, device=DEV)
        v = torch.zeros(pages, kv_heads, dim, 16, dtype=torch.bfloat16, device=DEV)
        ops.norm_qkv_rope_store(None, None, 1e-5, w, q, pos, seg, tables, cos, sin, k, v, heads, kv_heads, dim, dim, 16, prepared=prepared)
        return q, k, v

    plain = product()
    assert ops.tile_for_decode(w)
    for a, b in zip(plain, product()):
        assert torch.equal(a, b)
