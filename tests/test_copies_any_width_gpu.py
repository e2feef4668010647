"""Products of up to 16 rows from the tile-major copies of matrices of any width in steps of 32: every epilogue and prologue, tiles of 16 and
of 8 rows (both halves of a copied tile, a last one that is not whole), K ranges of the waves that are no whole blocks of 128 columns and ranges
that end early, activations staged and read where they lie.  The copy holds the same numbers and the launch multiplies them in the same
order, so all forms but two give the same bits as without it; the two that take whole tiles where there is a copy are held against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from fllm_amd.kernels import Ops
    return Ops()


def draw(shape, seed, scale=1.0, dtype=BF16):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(dtype).to(DEV)


# K: whole steps of 32 in every way eight (and sixteen) waves share them out; N: fewer tiles than half of the compute units, as many as fill
# them unevenly, more than are read where they lie
@pytest.mark.parametrize("M", [1, 7, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(16, 256), (40, 288), (1000, 544), (1536, 1536), (6150, 1568), (1528, 8960), (16500, 1056), (96, 13312)])
def test_plain_products(ops, M, N, K):
    x, w, bias = draw((M, K), M + K), draw((N, K), N + K, K ** -0.5), draw((N,), N, 0.3, torch.float32)
    start = draw((M, N), 5, 1.0, torch.float32)
    exact = x.double() @ w.double().T + bias.double()

    def forms():
        stored = ops.linear(x, w, torch.empty(M, N, dtype=BF16, device=DEV), bias=bias)
        added = ops.linear(x, w, start.clone(), bias=bias, accumulate=True)
        squared = torch.empty(M, N, dtype=BF16, device=DEV)
        assert ops.linear_relu_squared(x, w, squared)
        return stored, added, squared, ops.linear(x, w, torch.empty(M, N, device=DEV), bias=bias)

    plain = forms()
    assert ops.tile_for_decode(w)
    tiled = forms()
    for a, b in zip(plain[:3], tiled[:3]):
        assert torch.equal(a, b)
    # sums of K products of about K^-1/2: float32 rounding errors of K additions, in any order, stay far below this
    torch.testing.assert_close(tiled[3].double(), exact, rtol=0, atol=2.0 ** -24 * K ** 0.5 * 16)
    torch.testing.assert_close(tiled[0].double(), exact, rtol=2.0 ** -8, atol=1e-5)


@pytest.mark.parametrize("M", [1, 8, 12])
@pytest.mark.parametrize("N,K", [(48, 256), (1216, 1536), (4600, 2080), (17920, 1536)])
def test_behind_a_norm(ops, M, N, K):
    x, nw = draw((M, K), M, 2.0, torch.float32), draw((K,), K, 0.1, torch.float32) + 1
    w = draw((N, K), N, K ** -0.5)

    def forms():      # of the matrix `w` of the moment
        wide = ops.norm_linear(x, nw, 1e-5, w, torch.empty(M, N, dtype=BF16, device=DEV))
        gated = ops.norm_gate_up_glu(x, nw, 1e-5, w, torch.empty(M, N // 2, dtype=BF16, device=DEV), 7.0, 1.7, 1.0)
        swi = ops.norm_gate_up_swiglu(x, nw, 1e-5, w, torch.empty(M, N // 2, dtype=BF16, device=DEV))
        glu = ops.gate_up_glu(x.to(BF16), w, torch.empty(M, N // 2, dtype=BF16, device=DEV), 7.0, 1.7, 1.0)
        return wide, gated, swi, glu

    plain = forms()
    assert ops.tile_for_decode(w)
    assert torch.equal(plain[0], forms()[0])
    w = w.clone()
    assert ops.tile_for_decode(w, gate_up=True)
    for a, b in zip(plain, forms()):
        assert torch.equal(a, b)


# 16-row tiles from just beyond a tile for every other slot (of 512) to just short of two a slot; K whose halves are whole blocks of 128
# columns and not, whose last waves have nothing, and beyond what leaves room for both halves' sums in LDS (3,968) or for eight waves (4,512)
@pytest.mark.parametrize("M", [1, 8])
@pytest.mark.parametrize("N,K", [(4112, 256), (6150, 288), (8176, 1024), (8208, 1056), (16360, 544), (4600, 3008), (4600, 3968), (6144, 4512)])
def test_whole_tiles_of_a_copy_add_as_tiles_of_8_rows(ops, M, N, K):
    x, w, nw = draw((M, K), M + K), draw((N, K), N + K, K ** -0.5), draw((K,), K, 0.1, torch.float32) + 1

    def forms():
        squared = torch.empty(M, N, dtype=BF16, device=DEV)
        assert ops.linear_relu_squared(x, w, squared)
        return (ops.linear(x, w, torch.empty(M, N, dtype=BF16, device=DEV)), squared,
                ops.norm_linear(x.float(), nw, 1e-5, w, torch.empty(M, N, dtype=BF16, device=DEV)))

    plain = forms()
    assert ops.tile_for_decode(w)
    assert all(torch.equal(a, b) for a, b in zip(plain, forms()))


def test_what_is_read_beside_the_copy_stays_accepted(ops):
    """Rows that begin off 16 bytes have no 16-byte loads: they take the plain kernel, copy or not; a matrix that does gets no copy."""
    w = draw((64, 512), 1)
    assert ops.tile_for_decode(w)
    x = draw((3 * 512 + 1,), 2)[1:].view(3, 512)
    out = ops.linear(x, w, torch.empty(3, 64, dtype=BF16, device=DEV))
    torch.testing.assert_close(out.double(), x.double() @ w.double().T, rtol=2.0 ** -8, atol=1e-4)
    assert not ops.tile_for_decode(draw((64 * 512 + 1,), 3)[1:].view(64, 512))


def test_copies_that_begin_off_16_bytes_are_refused(ops):
    """A lane's load of a copy is 16 bytes: every entry point that takes one says so before it launches anything."""
    M, K, heads, dim = 4, 512, 2, 64
    p = lambda t: t.data_ptr()
    x, xb, nw = torch.zeros(M, K, device=DEV), torch.zeros(M, K, dtype=BF16, device=DEV), torch.ones(K, device=DEV)
    w, out = torch.zeros(3 * heads * dim, K, dtype=BF16, device=DEV), torch.zeros(M, 3 * heads * dim, device=DEV)
    rows, table = torch.zeros(M, dtype=torch.int32, device=DEV), torch.zeros(1, dtype=torch.float32, device=DEV)
    copy = torch.zeros(w.numel() + 8, dtype=BF16, device=DEV)
    tiles = p(copy) + 8
    N, lib, stream = w.shape[0], ops.lib, ops._stream()
    calls = {
        "norm_linear": lambda: lib.fllm_norm_linear(p(x), p(nw), 1e-5, p(w), tiles, None, p(out), M, N, K, stream),
        "norm_gate_up_swiglu": lambda: lib.fllm_norm_gate_up_swiglu(p(x), p(nw), 1e-5, p(w), tiles, None, p(out), M, N // 2, K, stream),
        "norm_gate_up_glu": lambda: lib.fllm_norm_gate_up_glu(p(x), p(nw), 1e-5, p(w), tiles, None, p(out), M, N // 2, K, 7.0, 1.7, 1.0, stream),
        "gate_up_glu": lambda: lib.fllm_gate_up_glu(p(xb), K, p(w), tiles, None, p(out), M, N // 2, K, 7.0, 1.7, 1.0, stream),
        "linear_relu_squared": lambda: lib.fllm_linear_relu_squared(p(xb), K, p(w), tiles, p(out), M, N, K, stream),
        "norm_qkv_rope_store": lambda: lib.fllm_norm_qkv_rope_store(p(x), p(nw), 1e-5, p(w), tiles, None, p(out), p(rows), p(rows), p(rows), 1, p(table),
                                                                    p(table), 0, None, None, M, heads, heads, dim, K, 16, 0, stream),
    }
    for name, call in calls.items():
        assert call() == -1, name
        assert b"aligned" in lib.fllm_last_error() or b"boundaries" in lib.fllm_last_error(), name


@pytest.mark.parametrize("M,K", [(16, 4608), (14, 5376)])
def test_a_shape_that_fits_no_plan_takes_the_general_kernel(ops, M, K):
    """More row tiles than there are counters for K slices, and more activations than LDS holds in one: such a matrix is served with a copy
    as it is without."""
    N = 262208
    w = (torch.randint(-8, 9, (N, K), device=DEV, dtype=torch.int8).to(BF16) * 2.0 ** -7)      # sums of whole multiples of 2^-14: exact
    x = (torch.randint(-8, 9, (M, K), device=DEV).to(BF16) * 2.0 ** -7)
    ends = torch.cat([torch.arange(3000), torch.arange(N - 3000, N)]).to(DEV)
    want = x.double() @ w[ends].double().T

    def forms():
        return (ops.linear(x, w, torch.empty(M, N, device=DEV)), ops.linear(x, w, torch.zeros(M, N, device=DEV), accumulate=True),
                ops.linear(x, w, torch.empty(M, N, dtype=BF16, device=DEV)))

    plain = forms()
    assert ops.tile_for_decode(w)
    for a, b in zip(plain, forms()):
        assert torch.equal(a, b)
    assert torch.equal(plain[0][:, ends].double(), want) and torch.equal(plain[1][:, ends].double(), want)


@pytest.mark.parametrize("M", [1, 8, 16, 40, 100])
@pytest.mark.parametrize("N,K", [(1000, 544), (1536, 1536), (6150, 1024)])
def test_plain_kernels_read_no_copy(M, N, K):
    """With the matrix-core kernels switched off a matrix with a copy gives the bits of one without: a chain of float32 sums a result."""
    from fllm_amd.kernels import Ops
    ops = Ops(library_gemm_from=None)
    x, w, start = draw((M, K), M + K), draw((N, K), N + K, K ** -0.5), draw((M, N), 5, 1.0, torch.float32)

    def forms():
        return (ops.linear(x, w, torch.empty(M, N, dtype=BF16, device=DEV)), ops.linear(x, w, torch.empty(M, N, device=DEV)),
                ops.linear(x, w, start.clone(), accumulate=True))

    ops.set_fast_kernels(False)
    try:
        plain = forms()
        assert ops.tile_for_decode(w)
        with_copy = forms()
    finally:
        ops.set_fast_kernels(True)
    assert all(torch.equal(a, b) for a, b in zip(plain, with_copy))


def test_copies_of_a_model_share_their_memory(ops):
    """Copies made together lie side by side, each on 256 bytes and whole, large ones in memory of their own; each goes with its matrix."""
    from fllm_amd.kernels import Ops
    ws = [draw((n, k), n + k) for n, k in ((16, 256), (40, 288), (1000, 544), (17, 1536))]
    wide = draw((4096, 40000), 7)
    gone = len(Ops._tiles)
    with ops.copies_together(sum(2 * w.numel() for w in ws)):
        for w in ws + [wide]:
            assert ops.tile_for_decode(w)
    tiles = [ops._tiles_of(w) for w in ws]
    assert len({t.untyped_storage().data_ptr() for t in tiles}) < len(ws) and all(t.data_ptr() % 256 == 0 for t in tiles)
    assert ops._tiles_of(wide).untyped_storage().nbytes() < 2 * wide.numel() + (2 << 20)
    alone = [w.clone() for w in ws]
    for w, t, other in zip(ws, tiles, alone):
        assert ops.tile_for_decode(other) and torch.equal(ops._tiles_of(other), t)
    assert len(Ops._tiles) == gone + 2 * len(ws) + 1
    del ws, wide, alone, w, other
    assert len(Ops._tiles) == gone


def test_copies_of_a_model_take_no_more_memory_than_theirs(ops):
    """Matrices of which the next does not fit behind the one before: what is allocated is what was made, and every byte is a copy's."""
    from fllm_amd.parts.runtime import Runtime
    rt = Runtime(torch.device(DEV), BF16, ops, 64, decode_weight_tiles=True)
    ws = [torch.zeros(n, k, dtype=BF16, device=DEV) for n, k in ((6001, 4096), (4096, 28672), (1544, 256), (6144, 4096), (4096, 28640))]
    rt.collect_tile_requests()
    for w in ws + [torch.zeros(64, 1000, dtype=BF16, device=DEV)]:      # the last has no copy
        rt.tile_for_decode(w)
    before = torch.cuda.memory_allocated()
    made = rt.tiles_for_model()
    assert made == sum(ops.copy_bytes(w) for w in ws)
    # torch's allocator hands out steps of 2 MiB from there on and keeps a remainder of up to 1 MiB with the block
    assert made <= torch.cuda.memory_allocated() - before <= made + len(ws) * (2 << 20)
    assert all(ops._tiles_of(w).numel() * 2 == ops.copy_bytes(w) for w in ws)


def test_copies_without_a_piece_lie_by_themselves(ops, monkeypatch):
    """No memory for the piece that copies were to share: each has its own, with the same contents; one that has none raises and leaves nothing."""
    import fllm_amd.kernels as kernels
    ws = [draw((48, 256), 1), draw((32, 512), 2)]
    total = sum(ops.copy_bytes(w) for w in ws)
    real, sizes = torch.empty, [total // 2]

    def empty(size, *args, **kwargs):
        if size in sizes:
            raise torch.cuda.OutOfMemoryError("no room")
        return real(size, *args, **kwargs)

    with monkeypatch.context() as m:
        m.setattr(kernels.torch, "empty", empty)
        with ops.copies_together(total):
            assert all(ops.tile_for_decode(w) for w in ws)
        lone = draw((64, 288), 3)
        sizes.append(ops.copy_bytes(lone) // 2)
        with pytest.raises(torch.cuda.OutOfMemoryError):
            ops.tile_for_decode(lone)
    assert ops._tiles_of(lone) is None
    tiles = [ops._tiles_of(w) for w in ws]
    assert tiles[0].untyped_storage().data_ptr() != tiles[1].untyped_storage().data_ptr()
    again = [w.clone() for w in ws]
    with ops.copies_together(total):
        assert all(ops.tile_for_decode(w) for w in again)
    together = [ops._tiles_of(w) for w in again]
    assert together[0].untyped_storage().data_ptr() == together[1].untyped_storage().data_ptr()
    assert all(torch.equal(a, b) for a, b in zip(tiles, together))
