"""Products of more than 64 bfloat16 rows whose operands the tile products do not take, through `Ops.linear`: rows that share memory (one row for all,
windows that overlap), products without a step or a column, with the kernels for matrix cores on and off; and float32 results on a stream
that is not the kernels'.  Float32 sums of K = 512 products of
bfloat16 operands that are exact in float64: K 2^-24 of the largest value, below 2^-14; bfloat16 results one rounding more, 2^-9."""
import pytest
import torch

pytestmark = pytest.mark.gpu
M, N, K = 96, 256, 512
FORMS = {"rows": lambda g: torch.randn(M, K, generator=g).bfloat16().cuda(),
         "one row": lambda g: torch.randn(1, K, generator=g).bfloat16().cuda().expand(M, K),
         "windows": lambda g: torch.randn(8 * M + K, generator=g).bfloat16().cuda().as_strided((M, K), (8, 1)),
         "odd windows": lambda g: torch.randn(M + K, generator=g).bfloat16().cuda().as_strided((M, K), (1, 1))}


@pytest.fixture
def ops():
    from fllm_amd.kernels import Ops
    ops = Ops()
    yield ops
    ops.set_fast_kernels(True)


@pytest.mark.parametrize("fast", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_operands_of_the_library(ops, dtype, fast):
    ops.set_fast_kernels(fast)
    g = torch.Generator().manual_seed(3)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    for form, made in FORMS.items():
        x, out = made(g), torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
        ops.linear(x, w, out)
        want = x.double() @ w.double().t()
        assert (out.double() - want).abs().max() <= (2.0 ** -14 if dtype == torch.float32 else 2.0 ** -8) * want.abs().max(), form
    nothing = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
    ops.linear(torch.empty(M, 0, dtype=torch.bfloat16, device="cuda"), torch.empty(N, 0, dtype=torch.bfloat16, device="cuda"), nothing)
    assert (nothing == 0).all()
    ops.linear(FORMS["rows"](g), torch.empty(0, K, dtype=torch.bfloat16, device="cuda"), torch.empty(M, 0, dtype=dtype, device="cuda"))


def test_float32_results_on_another_stream(ops):
    """The library has no workspace to share: such a product runs on any stream, also of a shape whose K the tiles cut on their own stream; nothing
    is asked of the device's stream for it."""
    from fllm_amd.kernels import Ops
    g = torch.Generator().manual_seed(4)
    x, w = torch.randn(1024, 8192, generator=g).bfloat16().cuda(), (torch.randn(2048, 8192, generator=g) * 8192 ** -0.5).bfloat16().cuda()
    want = x.double() @ w.double().t()
    ops._stream()
    claimed, other = dict(Ops._streams), torch.cuda.Stream()
    outs = [torch.full((1024, 2048), float("nan"), device="cuda") for _ in range(2)]
    ops.linear(x, w, outs[0])
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        ops.linear(x, w, outs[1])
    torch.cuda.synchronize()
    assert Ops._streams == claimed
    for out in outs:
        assert (out.double() - want).abs().max() <= 2.0 ** -10 * want.abs().max()
    library = torch.empty_like(outs[1])
    torch.mm(x, w.t(), out_dtype=torch.float32, out=library)
    assert torch.equal(outs[1], library)


@pytest.mark.parametrize("rows,columns,K,taken", [(1100, 16384, 2048, 1), (513, 28672, 4096, 1), (1537, 10240, 8192, 1), (1536, 16384, 2048, 0), (1024, 24576, 4096, 0)])
def test_plain_products_leave_the_library_where_they_fill_their_rounds(ops, rows, columns, K, taken):
    """All of them have a last round of half tiles; the first three fill 0.54 to 0.66 of their rounds and are the library's (1: declined)."""
    x, w = torch.zeros(rows, K, dtype=torch.bfloat16, device="cuda"), torch.zeros(columns, K, dtype=torch.bfloat16, device="cuda")
    out = torch.ones(rows, columns, dtype=torch.bfloat16, device="cuda")
    assert ops.lib.fllm_linear_tiles(x.data_ptr(), K, w.data_ptr(), None, out.data_ptr(), columns, rows, columns, K, 0, 0, ops._stream()) == taken
    assert (out == taken).all()
