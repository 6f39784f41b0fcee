"""Attention of single tokens over cached latents (csrc_seq/latent_attn.hip: absorb, the split pass, the combine) against float64, at block and size
edges: more single tokens than a workgroup takes, portions between them, ranks around every instantiation, splits of no keys.

Bound, per token and head: fp32 sums of n terms are within n 2^-24 of the sums of the absolute terms; in bf16 the folded query is rounded once
(2^-8), so a score is off by at most D = max_j (2^-8 [bf16] + 4 (dim + rank) 2^-24) scale sum |q||w_uk||c_j|; all the weights then change by a factor
within e^(+-2 D), their exponentials and the halves that carry them by 2^-13 more, the output by that much of sum w |c| |w_uv| plus the fp32 sums of
(keys + rank) terms and the result's rounding (2^-8 bf16, half a step of 8 significant bits)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(lens, ctx, heads, dim, vdim, rank, dtype, single_only, mfma, n_splits, window=0, sink=True, gate=True):
    from zhilight_amd import seqops
    g = torch.Generator(device=DEV).manual_seed(heads + rank + len(lens))
    rand = lambda *s: torch.randn(*s, device=DEV, generator=g)
    seqs, page = [], 0
    for i, (n, pos0) in enumerate(zip(lens, ctx)):
        k = (pos0 + n + 63) // 64
        seqs.append((n, pos0, i, list(range(page + k - 1, page - 1, -1))))          # (pages in falling order)
        page += k
    b, T = seqops.RaggedBatch(seqs, 64, DEV), sum(lens)
    cache = rand(page, 64, rank).to(dtype)
    w_uk, w_uv = (rand(heads * dim, rank) * rank ** -0.5).to(dtype), (rand(heads * vdim, rank) * rank ** -0.5).to(dtype)
    q = rand(T, 3 + heads * (dim + 1))
    sk, scale = rand(heads) if sink else None, dim ** -0.5
    out = torch.full((T, heads * vdim), 7.0, device=DEV, dtype=dtype)
    got = seqops.latent_attention(q, 3, q if gate else None, 3 + heads * dim, w_uk, w_uv, sk, cache, b, scale, heads, dim, vdim, out=out,
                                  single_only=single_only, mfma=mfma, n_splits=n_splits, window=window)
    uk, uv, t = w_uk.double().view(heads, dim, rank), w_uv.double().view(heads, vdim, rank), 0
    for (n, pos0, _, pages) in seqs:
        rows = cache[torch.tensor(pages, device=DEV)].reshape(-1, rank).double()
        for i in range(n):
            if single_only and n > 1:
                assert bool((got[t] == 7.0).all())
            else:
                pos = pos0 + i
                c = rows[max(0, pos - window + 1) if window else 0:pos + 1]
                qh = q[t, 3:3 + heads * dim].double().view(heads, dim)
                s = torch.einsum("hd,hdr->hr", qh, uk) @ c.T * scale
                D = (torch.einsum("hd,hdr->hr", qh.abs(), uk.abs()) @ c.abs().T).amax(1) * scale * ((2.0 ** -8 if dtype == torch.bfloat16 else 0) + 4 * (dim + rank) * 2.0 ** -24)
                full = torch.cat([s, sk.double()[:, None]], 1) if sink else s
                w = torch.softmax(full, 1)[:, :s.shape[1]]
                gt = torch.sigmoid(q[t, 3 + heads * dim:].double())[:, None] if gate else 1.0
                ref = torch.einsum("hr,hvr->hv", w @ c, uv) * gt
                size = torch.einsum("hr,hvr->hv", w @ c.abs(), uv.abs()) * gt
                half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
                bound = size * (torch.expm1(2 * D)[:, None] + 2.0 ** -13 + 2 * (len(c) + rank) * 2.0 ** -24) * (1 + half) + half * ref.abs()
                err = (got[t].double().view(heads, vdim) - ref).abs()
                assert bool((err <= bound + 1e-30).all()), (t, float((err / bound).max()))
            t += 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, dim, vdim, rank", [(1, 16, 16, 8), (17, 24, 20, 64), (3, 128, 128, 72), (2, 130, 12, 136), (16, 64, 64, 256), (32, 128, 128, 512),
                                                    (5, 40, 33, 520), (2, 192, 128, 640), (2, 16, 16, 648), (2, 32, 16, 808), (3, 20, 16, 30), (2, 16, 16, 33)])
def test_sizes(heads, dim, vdim, rank, dtype):
    for n_splits in (None, 1, 7):
        _run([1] * 9, [0, 31, 32, 33, 63, 64, 130, 200, 5], heads, dim, vdim, rank, dtype, False, True, n_splits)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mfma", [True, False])
def test_portions_windows_and_options(mfma, dtype):
    lens, ctx = [1, 3, 1, 1, 9, 1, 1, 1, 1, 12, 1], [40, 0, 100, 0, 70, 31, 64, 300, 1, 0, 129]
    for single_only in (True, False):
        for window in (0, 33):
            _run(lens, ctx, 6, 32, 32, 64, dtype, single_only, mfma, None, window)
    _run(lens, ctx, 6, 32, 32, 64, dtype, True, mfma, 70, 0, False, False)
    _run([1], [3000], 4, 32, 48, 128, dtype, True, mfma, None)
    _run([1, 1], [700, 10], 4, 32, 48, 128, dtype, True, mfma, 600)
