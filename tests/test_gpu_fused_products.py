"""Linears with their residual or their gate in the product's epilogue (csrc/dense_gemm.hip, csrc_seq/seq_gemm.hip): the bits of the separate calls --
the same kernels form the sums in the same order, the epilogues take the same steps."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rand(*shape, g, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, device=DEV, generator=g) * scale).to(dtype)


# every block of rows of the streaming kernel, tiles of 8 and 16 outputs with ragged ends, more tiles than workgroups; each tile shape of the large
# products, whole and ragged
SIZES = [(1, 16, 64), (2, 7, 128), (3, 2304, 320), (4, 4100, 128), (8, 1000, 1088), (9, 50, 512), (16, 4097, 192), (32, 129, 2304), (33, 64, 64), (77, 201, 1088),
         (257, 513, 64), (385, 1000, 64), (777, 5760, 128), (565, 10750, 64), (565, 4096, 128), (1024, 6144, 128), (2100, 4104, 64)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m, n, k", SIZES)
def test_dense_linear(m, n, k, dtype):
    from zhilight_amd import ops
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x, w, w2 = _rand(m, k, g=g, dtype=dtype), _rand(n, k, g=g, dtype=dtype, scale=k ** -0.5), _rand(n, k, g=g, dtype=dtype, scale=k ** -0.5)
    b, b2, res = _rand(n, g=g, dtype=dtype), _rand(n, g=g, dtype=dtype), _rand(m, n, g=g, dtype=dtype)
    assert ops.dense_linear_ok(x, w) and ops.dense_linear_ok(x, w, w2)

    def product(w, b):                                           # the plain product of the same kernel
        return ops.dense_linear(x, w, b)
    if m <= 32:
        assert torch.equal(product(w, b), ops.gemm_nt_small_m(x, w, bias=b))
    elif k % 128 == 0:
        assert torch.equal(product(w, b), ops.gemm_nt(x, w, bias=b))
    for bias in (None, b):
        for scale, whole in ((1.0, True), (0.2214, False)):
            got = res.clone()
            ops.dense_linear(x, w, bias, addend=got, scale=scale, scale_residual=whole, out=got)
            assert torch.equal(got, ops.element_add_scale(res, product(w, bias), scale, whole))
    for act in ("silu", "gelu"):
        for bias, bias2 in ((None, None), (b, b2)):
            assert torch.equal(ops.dense_linear(x, w, bias, up=w2, up_bias=bias2, act=act), ops.gate_mul(product(w, bias), product(w2, bias2), act))
    if 2 <= m <= 4:
        nw = _rand(k, g=g, dtype=dtype)
        parts = [ops.gemm_nt_small_m(x, v, norm_weight=nw, norm_eps=1e-5) for v in (w, w2)]
        got = ops.dense_linear(x, w, up=w2, norm_weight=nw)
        assert torch.equal(got, ops.gate_mul(*parts))
        assert torch.equal(ops.dense_linear(x[:1], w, up=w2, norm_weight=nw), got[:1])


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("m, ff, k", [s for s in SIZES if s[0] != 33] + [(700, 513, 64), (3, 40, 100), (40, 100, 2048)])
def test_gated_product_of_the_ragged_engine(m, ff, k, bias):
    from zhilight_amd import seqops
    g = torch.Generator(device=DEV).manual_seed(m + ff + k)
    wide, w = _rand(m, k + 8, g=g, dtype=torch.bfloat16), _rand(2 * ff, k, g=g, dtype=torch.bfloat16, scale=k ** -0.5)
    b = _rand(2 * ff, g=g) if bias else None
    for x in (wide[:, :k], wide[:, 3:k + 3]):                    # (the second: rows that are not 16-byte aligned, the separate calls)
        for kind in ("silu", "gelu_tanh"):
            z = seqops.gemm_nt(x, w, bias=b)
            assert torch.equal(seqops.gated_product(x, w, kind, b), seqops.act_mul(z, torch.bfloat16, kind=kind))


def test_what_the_kernels_do_not_take_is_refused():
    from zhilight_amd import ops
    x, w = torch.zeros(20, 96, dtype=torch.float16, device=DEV), torch.zeros(64, 96, dtype=torch.float16, device=DEV)
    assert not ops.dense_linear_ok(x, w)
    with pytest.raises(ops.ZLError):
        ops.dense_linear(x, w)
    with pytest.raises(ops.ZLError):
        ops.dense_linear(torch.zeros(5, 64, dtype=torch.float16, device=DEV), w[:, :64].contiguous(), norm_weight=torch.ones(64, dtype=torch.float16, device=DEV))
