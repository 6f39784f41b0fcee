"""Products of a few rows on the streaming kernel (csrc/zl_stream16.h), through both libraries, against the float64 product.

Bound: fp32 sums of k products (each wave adds its share in order, the waves' shares are added): k 2^-24 sum|x||w|, plus the result's rounding."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
HALF_ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}


def _operands(m, n, k, dtype):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    return torch.randn(m, k, device=DEV, generator=g).to(dtype), torch.randn(n, k, device=DEV, generator=g).mul_(k ** -0.5).to(dtype)


def _check(y, x, w, extra=0.0):
    xd, wd = x.double(), w.double()
    ref = xd @ wd.T + extra
    bound = HALF_ULP[y.dtype] * ref.abs() * 1.01 + x.shape[1] * 2.0 ** -24 * (xd.abs() @ wd.abs().T) + 1e-7
    assert bool(((y.double() - ref).abs() <= bound).all())


# fewer slices than waves, one tile, ragged last tiles, more tiles than workgroups, every block of rows of x and its edges
SIZES = [(1, 16, 64), (1, 5000, 320), (2, 40, 64), (3, 33, 576), (4, 4100, 128), (4, 7, 8192), (5, 1000, 1088), (8, 4113, 256), (9, 50, 512), (16, 4097, 192),
         (17, 16, 64), (32, 4112, 704), (31, 129, 2304)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m, n, k", SIZES)
def test_few_rows(m, n, k, dtype):
    from zhilight_amd import ops
    x, w = _operands(m, n, k, dtype)
    _check(ops.gemm_nt_small_m(x, w), x, w)
    bias = torch.randn(n, device=DEV).to(dtype)
    _check(ops.gemm_nt_small_m(x, w, bias=bias, alpha=0.5), x * 0.5, w, bias.double())


@pytest.mark.parametrize("m, n, k", SIZES)
def test_few_rows_on_the_ragged_engine(m, n, k):
    from zhilight_amd import seqops
    x, w = _operands(m, n, k, torch.bfloat16)
    _check(seqops.gemm_nt(x, w), x, w)
    bias = torch.randn(n, device=DEV)
    y, y2 = seqops.gemm_nt(x, w, bias=bias, lead=n // 2 + 1)
    _check(y, x, w, bias.double())
    assert torch.equal(y2, y[:, :n // 2 + 1].to(torch.bfloat16))
    z = seqops.gemm_nt(x, w, out_dtype=torch.bfloat16)
    _check(z, x, w)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m, n, k", [(2, 100, 64), (3, 4200, 2304), (4, 1000, 8192)])
def test_norm_on_the_way_in(m, n, k, dtype):
    """the rows that the stand-alone norm leaves, then the product (the sum of squares is added in another order: a value in a few hundred may round to
    its neighbour, which moves a sum by at most an ulp of that value times its weight: within the bound's k terms times 2^-8 here)"""
    from zhilight_amd import ops
    x, w = _operands(m, n, k, dtype)
    nw = (1 + 0.1 * torch.randn(k, device=DEV)).to(dtype)
    xn = ops.rmsnorm(x, nw, 1e-5)
    got, want = ops.gemm_nt_small_m(x, w, norm_weight=nw, norm_eps=1e-5).double(), xn.double() @ w.double().T
    assert bool(((got - want).abs() <= 2 * HALF_ULP[dtype] * (want.abs() + (xn.double().abs() @ w.double().abs().T) * 0.1)).all())


@pytest.mark.parametrize("m, n", [(2, 17), (3, 5000), (4, 128256)])
def test_greedy_pick(m, n):
    """the first of the largest rounded values of every row, ties within and between workgroups"""
    from zhilight_amd import ops
    x, w = _operands(m, n, 128, torch.float16)
    w[n // 3] = w[n - 1]
    ws = ops.argmax_workspace(m, n, DEV)
    y = ops.gemm_nt_small_m(x, w, argmax_ws=ws)
    tokens = torch.full((m,), -1, dtype=torch.int32, device=DEV)
    ops.greedy_advance(ws, m, n, tokens=tokens)
    first = (y == y.max(1, keepdim=True).values).to(torch.int8).argmax(1)
    assert torch.equal(tokens.long(), first)
