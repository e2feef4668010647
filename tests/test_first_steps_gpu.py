"""What a request's first step does beside a model's layers: slots of state tensors cleared in one launch."""
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
