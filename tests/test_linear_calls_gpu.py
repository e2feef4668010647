"""Products of more than 64 bfloat16 rows whose operands the tile products do not take, through `Ops.linear`: rows that share memory (one row for all,
windows that overlap), products without a step or a column, with the kernels for matrix cores on and off.  Float32 sums of K = 512 products of
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
