"""What a request's first steps do beside a model's layers: slots of state tensors cleared in one launch; the gate of a token's side input
for the rows of a busy step."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


def test_cleared_slots_and_no_others(ops):
    """Tensors of several types, slots of a few bytes that begin anywhere and of more than a workgroup clears, more slots than a launch names."""
    shapes = [((70, 3), torch.bfloat16), ((70, 1), torch.int8), ((70, 5, 7), torch.float32), ((70, 33, 257), torch.float32), ((90, 16384 + 3), torch.bfloat16),
              ((70, 17), torch.int8)]
    tensors = [torch.ones(s, dtype=d, device=DEV) for s, d in shapes]
    table = ops.slot_table(tensors)
    ops.clear_slots(table, [])
    assert all(bool((t == 1).all()) for t in tensors)
    for slots in ([3], [0, 69, 8], [s for s in range(70) if s % 11 != 4]):
        for t in tensors:
            t.fill_(1)
        ops.clear_slots(table, slots)
        for t in tensors:
            want = torch.ones_like(t)
            want[slots] = 0
            assert torch.equal(t, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17, 32])
def test_side_gate_of_more_rows(ops, rows, dtype):
    """Eight rows a workgroup: a row's numbers are those of its own call, whichever rows it comes with."""
    g = torch.Generator().manual_seed(rows)
    width, dim = 520, 24
    x, w = (torch.randn(rows, width, generator=g) * 3).to(DEV), (torch.randn(dim, width, generator=g) * width ** -0.5).to(dtype).to(DEV)
    table, ids = torch.randn(31, 3 * dim, generator=g).to(dtype).to(DEV), torch.randint(0, 31, (rows,), generator=g, dtype=torch.int32).to(DEV)
    got = torch.full((rows, dim), float("nan"), dtype=dtype, device=DEV)
    assert ops.side_gate_rows(x, w, ids, table, dim, got)
    alone = torch.empty_like(got)
    for r in range(rows):
        assert ops.side_gate(x[r:r + 1], w, ids[r:r + 1], table, dim, alone[r:r + 1])
    assert torch.equal(got, alone)
    assert not ops.side_gate_rows(torch.zeros(33, width, device=DEV), w, torch.zeros(33, dtype=torch.int32, device=DEV), table, 0,
                                  torch.empty(33, dim, dtype=dtype, device=DEV))


def test_side_gate_of_more_rows_is_left_to_the_plain_product_where_that_is_asked_for(ops):
    x, w = torch.zeros(9, 64, device=DEV), torch.zeros(8, 64, dtype=torch.bfloat16, device=DEV)
    ids, table = torch.zeros(9, dtype=torch.int32, device=DEV), torch.zeros(4, 8, dtype=torch.bfloat16, device=DEV)
    out = torch.empty(9, 8, dtype=torch.bfloat16, device=DEV)
    ops.set_fast_kernels(False)
    try:
        assert not ops.side_gate_rows(x, w, ids, table, 0, out)
        assert ops.side_gate(x[:8], w, ids[:8], table, 0, out[:8])
    finally:
        ops.set_fast_kernels(True)
    assert ops.side_gate_rows(x, w, ids, table, 0, out)
