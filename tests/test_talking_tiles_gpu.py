"""Row tiles of the attention whose heads talk to each other, at the edges of its blocks of 128 keys: the instances that are built for a
head count and the general one, shares of a tile's blocks (more blocks than the caller's bound allows for among them), pages that are a power
of two, a multiple of eight and of four, value widths that leave waves without lanes of their own, chunks that end inside a tile."""
import pytest
import torch

from reference_ops import ReferenceOps
from test_menitar_gpu import BF16_EPS, DEV, Scene, close, run_mixer_kernels

pytestmark = pytest.mark.gpu

# heads, kv heads, key size, value size, chunk, page
SHAPES = [(8, 2, 128, 128, None, 16), (12, 2, 128, 128, 300, 64), (16, 2, 128, 80, 130, 8), (12, 2, 128, 112, None, 4), (16, 2, 128, 128, 140, 24),
          (15, 3, 192, 48, None, 12), (16, 16, 160, 16, 200, 16), (7, 7, 96, 128, 129, 32), (8, 4, 256, 96, None, 8)]
# every instance built for a head count on 1, 2 or 4 key/value heads of 128 lanes, values of 80 to 128, pages of 8 to 64
SHAPES += [(H, G, 128, (128, 80, 96, 112)[(H // 2 + G) % 4], (None, 130, 200)[(H + G) % 3], (8, 16, 32, 64)[(H // 2 + G // 2) % 4])
           for G in (1, 2, 4) for H in range(4, 17, 2) if H % G == 0 and (G, H) not in ((2, 8), (2, 12), (2, 16))]
# (held, new): tiles of one row to several, last keys right before, on and behind a block's edge
SEGMENTS = [(0, 129), (111, 17), (112, 16), (127, 2), (254, 3), (383, 33), (0, 5), (500, 12)]


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


@pytest.mark.parametrize("splits", [1, 2, 4])
@pytest.mark.parametrize("shape", SHAPES)
def test_blocks_of_128_keys(ops, shape, splits):
    H, G, d, dv, chunk, page = shape
    ref, scale = ReferenceOps(), d ** -0.5
    loud = [(s, held + new, 8.0) for s, (held, new) in enumerate(SEGMENTS)]      # the slot behind a request's last token
    sc = Scene(SEGMENTS, H, G, d, dv, page, 32, seed=H + d + dv, dtype=torch.bfloat16, loud=loud)
    for s, (held, new) in enumerate(SEGMENTS):                                   # and what lies in it for the values
        at = held + new
        sc.v_pages[int(sc.tables[s, at // page]), :, :, at % page] = float("nan")
    t = sc.tensors(DEV)
    if splits == 4:      # fewer blocks than the rows see: shares still cover all of them
        sc.max_pos = 64
    q, got = run_mixer_kernels(ops, t, sc, chunk, scale, torch.bfloat16, splits)
    torch.cuda.synchronize()
    # the reference goes on from the queries, keys and values that the store kernel left (its own test holds those)
    w = {n: v.cpu().double() if v.dtype in (torch.bfloat16, torch.float32) else v.cpu() for n, v in t.items()}
    want = torch.empty(got.shape, dtype=torch.float64)
    gate_at = H * d + G * (d + dv)
    ref.talking_attention(q.cpu().double(), w["qkvg"][:, gate_at:gate_at + H], w["k_pages"], w["v_pages"].nan_to_num(0.0), w["tables"],
                          w["row_pos"], w["row_seg"], w["seg_start"], w["talk"], w["temp"], want, H, G, d, dv, page, scale, chunk, 8, 600)
    # weights and the result are rounded to bfloat16 (2^-9 of each), scores of up to about 30 carry float32 sums
    close(got, want, 3 * BF16_EPS, 3e-2, "attention")


# heads, kv heads, key size, value size, chunk, page: the instances for up to two, four and eight key/value heads of 128 lanes, and beside their rule
SINGLE = [(12, 2, 128, 128, None, 16), (16, 1, 128, 128, 100, 8), (5, 1, 128, 128, None, 64), (12, 2, 128, 128, 70, 24), (9, 3, 128, 128, None, 16),
          (16, 8, 64, 128, 130, 16), (6, 2, 128, 112, None, 32), (12, 4, 128, 128, None, 16), (8, 4, 128, 128, 100, 8), (16, 8, 128, 128, None, 64),
          (12, 6, 128, 128, 130, 16)]


@pytest.mark.parametrize("splits", [1, 2, 4])
@pytest.mark.parametrize("shape", SINGLE)
def test_single_rows(ops, shape, splits):
    """Contexts around a block of 64 keys and several blocks a workgroup, with what is no number behind the last token."""
    H, G, d, dv, chunk, page = shape
    ref, scale = ReferenceOps(), d ** -0.5
    sc = Scene([(n, 1) for n in (0, 15, 62, 63, 64, 99, 127, 128, 300, 511)], H, G, d, dv, page, 32, seed=H + d + dv, dtype=torch.bfloat16)
    for s in range(10):
        at = int(sc.row_pos[s]) + 1
        sc.v_pages[int(sc.tables[s, at // page]), :, :, at % page] = float("nan")
        sc.k_pages[int(sc.tables[s, at // page]), :, :, at % page] *= 8.0
    t = sc.tensors(DEV)
    q, got = run_mixer_kernels(ops, t, sc, chunk, scale, torch.bfloat16, splits, single_rows=True)
    torch.cuda.synchronize()
    w = {n: v.cpu().double() if v.dtype in (torch.bfloat16, torch.float32) else v.cpu() for n, v in t.items()}
    want = torch.empty(got.shape, dtype=torch.float64)
    gate_at = H * d + G * (d + dv)
    ref.talking_attention(q.cpu().double(), w["qkvg"][:, gate_at:gate_at + H], w["k_pages"], w["v_pages"].nan_to_num(0.0), w["tables"],
                          w["row_pos"], w["row_seg"], w["seg_start"], w["talk"], w["temp"], want, H, G, d, dv, page, scale, chunk, 8, 600)
    close(got, want, 3 * BF16_EPS, 3e-2, "attention")      # the same roundings as the tiles'
