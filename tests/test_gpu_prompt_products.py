"""Products of prompt portions on the large tiles (csrc/zl_gemm16.h), through both libraries, against the float64 product of the same numbers.

Bound: the sums are fp32 in k order, so they are within k 2^-24 sum|x||w| of the exact ones (every partial sum is at most sum|x||w|), and the
result carries one rounding to its format (2^-11 fp16, 2^-8 bf16, each half an ulp)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
HALF_ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}


def _operands(m, n, k, dtype, ldx=None, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(m, ldx or k, device=DEV, generator=g).to(dtype)[:, :k]
    w = torch.randn(n, k, device=DEV, generator=g).mul_(k ** -0.5).to(dtype)
    return x, w


def _check(y, x, w, extra=0.0):
    xd, wd = x.double(), w.double()
    ref = xd @ wd.T + extra
    bound = HALF_ULP[y.dtype] * ref.abs() + x.shape[1] * 2.0 ** -24 * (xd.abs() @ wd.abs().T) + 1e-7
    off = (y.double() - ref).abs()
    assert bool((off <= bound).all()), float((off / bound).max())


# 256 x 256, 256 x 128, 128 x 128 in rounds, 128 x 128 alone, 128 x 64 and 64 x 64 tiles, each with whole tiles and with ragged edges
SIZES = [(4096, 4096, 128), (2100, 8200, 64), (1024, 6144, 192), (1000, 6100, 192), (2048, 3072, 128), (2040, 3075, 64), (1280, 2048, 320), (1153, 2047, 64),
         (512, 1280, 640), (385, 1000, 64), (33, 64, 64), (64, 128, 128), (77, 201, 1088), (257, 513, 64)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m, n, k", SIZES)
def test_dense_product(m, n, k, dtype):
    from zhilight_amd import ops
    k = (k + 127) // 128 * 128                                   # (this library's rows are whole 128s)
    x, w = _operands(m, n, k, dtype)
    bias = torch.randn(n, device=DEV).to(dtype)
    _check(ops.gemm_nt(x, w), x, w)
    _check(ops.gemm_nt(x, w, bias=bias, alpha=0.5), x * 0.5, w, bias.double())


@pytest.mark.parametrize("m, n, k", SIZES)
def test_ragged_engine_product(m, n, k):
    from zhilight_amd import seqops
    x, w = _operands(m, n, k, torch.bfloat16, ldx=k + 8)
    _check(seqops.gemm_nt(x, w), x, w)
    _check(seqops.gemm_nt(x, w, out_dtype=torch.bfloat16), x, w)
    bias = torch.randn(n, device=DEV)
    lead = n // 2
    y, y2 = seqops.gemm_nt(x, w, bias=bias, lead=lead)
    _check(y, x, w, bias.double())
    assert torch.equal(y2, y[:, :lead].to(torch.bfloat16))


@pytest.mark.parametrize("m, n, k", [(40, 200, 2048), (100, 2048, 8192), (17, 64, 576), (65, 130, 1088)])
def test_ragged_engine_product_with_a_divided_k(m, n, k):
    from zhilight_amd import seqops
    assert seqops._k_parts(m, n, k) > 1
    x, w = _operands(m, n, k, torch.bfloat16)
    _check(seqops.gemm_nt(x, w), x, w)


def test_a_row_that_is_not_finite_stays_alone():
    from zhilight_amd import ops, seqops
    x, w = _operands(200, 200, 256, torch.bfloat16)
    x[199], x[64] = float("nan"), float("inf")
    for y in (ops.gemm_nt(x, w), seqops.gemm_nt(x, w)):
        rows = torch.isfinite(y).all(1)
        assert not rows[199] and not rows[64] and int(rows.sum()) == 198
