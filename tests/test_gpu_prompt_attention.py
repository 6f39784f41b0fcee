"""Portions on the ragged engine's attention kernels at sizes where their work is shared out differently: query tiles of two groups of waves, key tiles
in part hidden by the causal edge or a window, heads that are no whole 8s, few and many output blocks -- against float64 softmax attention.

Bound: queries and weights reach the matrix cores as bf16 (latent: the query once, 2^-8; window: both halves, 2^-16; weights: both halves, 2^-15), so a score
is off by at most D = (2^-8 or 2^-15) scale sum |q||k| and the weights by a factor within e^(+-2 D); exponentials, running sums and corrections add 2^-13, the
fp32 sums (keys + dim) 2^-23, the bf16 result 2^-8."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _batch(lens, ctx):
    from zhilight_amd import seqops
    seqs, page = [], 0
    for i, (n, pos0) in enumerate(zip(lens, ctx)):
        k = (pos0 + n + 63) // 64
        seqs.append((n, pos0, i, list(range(page + k - 1, page - 1, -1))))
        page += k
    return seqops.RaggedBatch(seqs, 64, DEV), seqs, page


def _softmax(q, k, v, pos, window, scale, sink):
    """q (H, d), k / v (keys, H, d): output and the sizes that the bound is made of"""
    lo = max(0, pos - window + 1) if window else 0
    k, v = k[lo:pos + 1], v[lo:pos + 1]
    s = torch.einsum("hd,khd->hk", q, k) * scale
    qk = (torch.einsum("hd,khd->hk", q.abs(), k.abs()) * scale).amax(1)
    full = torch.cat([s, sink[:, None]], 1) if sink is not None else s
    w = torch.softmax(full, 1)[:, :s.shape[1]]
    return torch.einsum("hk,khd->hd", w, v), torch.einsum("hk,khd->hd", w, v.abs()), qk


def _check(got, ref, size, qk, unit, keys, dim):
    bound = size * (torch.expm1(2 * unit * qk)[:, None] + 2.0 ** -13 + (keys + dim) * 2.0 ** -23) + 2.0 ** -8 * (ref.abs() + size * 2.0 ** -7)
    err = (got.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


# one workgroup per CU and less, pairs of groups, more than 1024 workgroups; every size of head
@pytest.mark.parametrize("lens, ctx", [((130, 2, 64), (0, 70, 1)), ((700,), (0,)), ((65, 300), (500, 0))])
@pytest.mark.parametrize("heads, dim, vdim, window", [(16, 128, 128, 0), (16, 128, 128, 200), (3, 64, 32, 0), (3, 60, 64, 100), (2, 128, 48, 0), (2, 192, 128, 64), (2, 100, 30, 0),
                                                      (1, 256, 256, 0), (130, 16, 16, 0)])
def test_latent_portions(heads, dim, vdim, window, lens, ctx):
    from zhilight_amd import seqops
    b, seqs, _ = _batch(lens, ctx)
    g = torch.Generator(device=DEV).manual_seed(heads + dim + sum(lens))
    rand = lambda *s: torch.randn(*s, device=DEV, generator=g)
    T, (start, pos0, _, n_ctx) = sum(lens), b.context(window)
    q = rand(T, heads * dim + heads + 4)
    k, v = rand(n_ctx, heads * dim).bfloat16(), rand(n_ctx, heads * vdim).bfloat16()
    vt = torch.zeros(heads * vdim, (n_ctx + 7) // 8 * 8, device=DEV, dtype=torch.bfloat16)
    vt[:, :n_ctx] = v.T
    sink, out, scale = rand(heads), torch.zeros(T, heads * vdim, device=DEV, dtype=torch.bfloat16), dim ** -0.5
    seqops.latent_attention_prompt(q, 4, q, 4 + heads * dim, k, vt, sink, b, scale, heads, dim, vdim, out, window=window)
    start, pos0, t = start.tolist(), None if pos0 is None else pos0.tolist(), 0
    for i, (n, p0, _, _) in enumerate(seqs):
        c0 = pos0[i] if pos0 else 0
        ks, vs = (x[start[i]:].double().view(-1, heads, d) for x, d in ((k, dim), (v, vdim)))
        for j in sorted({0, 1, 15, 16, 62, 63, 64, 65, n // 2, n - 2, n - 1}):
            if not 0 <= j < n:
                continue
            qh, gate = q[t + j, 4:4 + heads * dim].double().view(heads, dim), torch.sigmoid(q[t + j, 4 + heads * dim:].double())[:, None]
            ref, size, qk = _softmax(qh, ks, vs, p0 + j - c0, window, scale, sink.double())
            _check(out[t + j].view(heads, vdim), ref * gate, size * gate, qk, 2.0 ** -8, p0 + j + 1, dim)
        t += n


@pytest.mark.parametrize("heads, kv_heads, dim, vdim", [(16, 4, 128, 128), (4, 2, 64, 64), (4, 1, 40, 16), (2, 1, 96, 144), (2, 2, 128, 256), (1, 1, 256, 128)])
@pytest.mark.parametrize("window", [0, 100, 64])
def test_window_portions(heads, kv_heads, dim, vdim, window):
    from zhilight_amd import seqops
    lens, ctx = (130, 2, 300, 64), (0, 70, 33, 1)
    b, seqs, pages = _batch(lens, ctx)
    g = torch.Generator(device=DEV).manual_seed(heads + dim + vdim)
    rand = lambda *s: torch.randn(*s, device=DEV, generator=g)
    T, G = sum(lens), kv_heads
    kc, vc = rand(pages, 64, G, dim).bfloat16(), rand(pages, G, vdim, 64).bfloat16()
    q, scale = rand(T, 4 + heads * dim), dim ** -0.5
    acc, ml, ns = seqops.window_attention(q, 4, kc.view(pages, 64, -1), vc.view(pages, 64, -1), b, scale, window, heads, G, dim, vdim, all_kv=False)
    out = seqops.head_mix_gate(acc, ml, ns, None, None, None, 0, b, heads, G, vdim, torch.bfloat16)
    t = 0
    for n, p0, _, pg in seqs:
        rows = torch.tensor(pg, device=DEV)
        per = heads // G
        ks = kc[rows].reshape(-1, G, dim).double().repeat_interleave(per, 1)
        vs = vc[rows].permute(0, 3, 1, 2).reshape(-1, G, vdim).double().repeat_interleave(per, 1)
        for j in sorted({0, 1, 15, 16, 62, 63, 64, 65, n // 2, n - 2, n - 1}):
            if 0 <= j < n:
                qh = q[t + j, 4:].double().view(heads, dim)
                ref, size, qk = _softmax(qh, ks, vs, p0 + j, window, scale, None)
                _check(out[t + j].view(heads, vdim), ref, size, qk, 2.0 ** -15, p0 + j + 1, dim)
        t += n
