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


# 256 x 256, 256 x 128, 128 x 128 in rounds, 128 x 128 alone, 128 x 64 and 64 x 64 tiles, each with whole tiles and with ragged edges; 160 x 128,
# 192 x 128 and 160 x 64 tiles
SIZES = [(4096, 4096, 128), (2100, 8200, 64), (1024, 6144, 192), (1000, 6100, 192), (2048, 3072, 128), (2040, 3075, 64), (1280, 2048, 320), (1153, 2047, 64),
         (512, 1280, 640), (385, 1000, 64), (33, 64, 64), (64, 128, 128), (77, 201, 1088), (257, 513, 64),
         (800, 11520, 64), (777, 11460, 192), (576, 21504, 64), (565, 21440, 64), (640, 4096, 128), (565, 4090, 320), (640, 11520, 64), (513, 11516, 128), (193, 4099, 64), (1000, 5100, 64)]


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


# ---- prompt attention of 64-wide heads (csrc/prefill_attn.hip, zl_prefill_attn_w32) -----------------------------------------------------
def _attention64(q, k, v, pos0, scale):
    s, h, d = q.shape
    g = k.shape[1]
    kd, vd = (t[:pos0 + s].double().repeat_interleave(h // g, 1).transpose(0, 1) for t in (k, v))
    sc = (q.double().transpose(0, 1) @ kd.transpose(1, 2)) * scale
    seen = torch.arange(pos0 + s, device=DEV)[None, :] <= pos0 + torch.arange(s, device=DEV)[:, None]
    return (torch.softmax(sc.masked_fill(~seen, float("-inf")), -1) @ vd).transpose(0, 1)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("s, pos0, h, g, bshd", [(1, 0, 1, 1, True), (16, 0, 4, 2, False), (17, 63, 3, 3, True), (63, 1, 2, 1, True), (64, 64, 2, 2, False),
                                                 (65, 0, 36, 36, True), (200, 129, 6, 2, True), (777, 0, 4, 4, True)])
def test_prompt_attention_of_64_wide_heads(s, pos0, h, g, bshd, dtype):
    """Bound: probabilities carry 2^-16 (bf16) and better, the exponent of a score of magnitude S is off by S 2^-22 at most (fp32 sums of 64
    products, one multiply, the hardware's exp2): 1e-4 of the largest value here, plus the result's own rounding."""
    from zhilight_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(s + pos0)
    n = pos0 + s + 7
    q = torch.randn(s, h, 64, device=DEV, generator=gen).to(dtype)
    k, v = (torch.randn(n, g, 64, device=DEV, generator=gen).to(dtype) for _ in range(2))
    k[pos0 + s:], v[pos0 + s:] = float("nan"), float("inf")     # slots that no query sees hold anything
    ref = _attention64(q, k, v, pos0, 0.125)
    lay = (lambda t: t) if bshd else (lambda t: t.transpose(0, 1).contiguous())
    out = ops.prefill_attention_w32(q, lay(k), lay(v), pos0, g, 0.125, bshd=bshd)
    assert bool(((out.double() - ref).abs() <= HALF_ULP[dtype] * ref.abs() + 1e-4 * float(ref.abs().max())).all())


def test_prompt_attention_of_64_wide_heads_keeps_later_values_out():
    """a value that is not finite reaches no block of 16 queries before its own"""
    from zhilight_amd import ops
    q, k, v = (torch.randn(128, 2, 64, device=DEV).to(torch.bfloat16) for _ in range(3))
    v[100] = float("inf")
    out = ops.prefill_attention_w32(q, k, v, 0, 2, 0.125)
    assert bool(torch.isfinite(out[:96]).all()) and not bool(torch.isfinite(out[100:]).any())
    for bad in (dict(d=128), dict(d=32)):
        from zhilight_amd._lib import ZLError
        with pytest.raises(ZLError):
            ops.prefill_attention_w32(*(torch.zeros(8, 2, bad["d"], device=DEV, dtype=torch.bfloat16) for _ in range(3)), 0, 2, 0.1)


# ---- INT8 linears of prompt chunks (zl_int8_linear): the bits of the separate calls -----------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m, n, k", [(33, 16, 128), (64, 100, 256), (100, 1001, 384), (257, 514, 128), (1000, 2048, 256), (1025, 6144, 128), (2049, 4100, 128)])
def test_int8_linear(m, n, k, dtype):
    from zhilight_amd import ops
    g = torch.Generator(device=DEV).manual_seed(m)
    a, b, b2 = (torch.randint(-127, 128, (r, k), device=DEV, generator=g, dtype=torch.int8) for r in (m, n, n))
    sx = torch.rand(m, device=DEV, generator=g) * 0.02
    sy, sy2 = (torch.rand(n, device=DEV, generator=g).mul(0.02).to(dtype) for _ in range(2))
    c, c2 = ((a.double() @ w.double().T).round().to(torch.int32) for w in (b, b2))
    assert torch.equal(ops.int8_gemm_nt(a, b), c)
    assert torch.equal(ops.int8_linear(a, sx, b, sy, dtype=dtype), ops.quant_scale_back(c, sx, sy, dtype))
    assert torch.equal(ops.int8_linear(a, sx, b, sy, b2, sy2, dtype=dtype), ops.quant_back_act_mul(c, sx, sy, c2, sx, sy2, "silu", dtype))
    add = torch.randn(m, n, device=DEV, generator=g).to(dtype)
    want = ops.quant_back_element_add_scale(c, sx, sy, add, 0.5)
    assert torch.equal(ops.int8_linear(a, sx, b, sy, addend=add, scale=0.5, out=add), want)


@pytest.mark.parametrize("rows, width", [(1, 8), (64, 512), (131, 576), (300, 24)])
def test_gathered_rows(rows, width):
    from zhilight_amd import seqops
    x = torch.randn(200, width, device=DEV).bfloat16()
    at = torch.randint(0, 200, (rows,), device=DEV, dtype=torch.int32)
    assert torch.equal(seqops.gather_rows(x, at), x[at.long()])
