"""Row steps that hold their numbers in registers, four to a lane, against float64: PolyNorm, the residual norms, token shift, embedding, the short
convolution, group norms and plain heads' gates -- and the loops that keep widths that are no multiple of 4 and unaligned rows.

Bound: a row's sum of squares (all terms >= 0) in any order of fp32 steps is off by less than (width / 256 + 16) 2^-24 of itself for the loops (a
thread adds width / 256 terms, then 8 lane steps and 16 waves) and less for the registers; half of it reaches the result.  Everything else is at most
16 roundings, and a bf16 result (8 significant bits: half a step is at most 2^-8 of the number) adds 2^-8:
|got - ref| <= ((width / 256 + 32) 2^-24 + 2^-8 [bf16]) * size, size = the sum of the absolute terms."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# the smallest; no multiple of 4; a piece's ends for 256 and 1024 threads; 2 and 8 pieces; beyond the registers
WIDTHS = [4, 6, 252, 260, 1024, 1028, 4096, 8196, 21504, 32768, 32772]


def _close(got, ref, size, width):
    eps = (width / 256 + 32) * 2.0 ** -24 + (2.0 ** -8 if got.dtype == torch.bfloat16 else 0.0)
    err = (got.double() - ref).abs()
    assert bool((err <= eps * size + 1e-30).all()), float((err / (eps * size + 1e-30)).max())


def _rand(*shape, g):
    return torch.randn(*shape, device=DEV, generator=g)


def _unaligned(t):
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    v = buf[1:].view(t.shape)
    v.copy_(t)
    return v


def _batch(lens):
    from zhilight_amd import seqops
    seqs, page = [], 0
    for i, n in enumerate(lens):
        k = (n + 63) // 64
        seqs.append((n, 0, len(lens) - i, list(range(page, page + k))))          # (slots in another order, slot 0 nobody's)
        page += k
    return seqops.RaggedBatch(seqs, 64, DEV)


@pytest.mark.parametrize("off", [False, True])
@pytest.mark.parametrize("rows", [1, 515])
@pytest.mark.parametrize("width", WIDTHS)
def test_row_norms(width, rows, off):
    from zhilight_amd import seqops
    if rows > 1 and width > 8196:
        rows = 3
    g = torch.Generator(device=DEV).manual_seed(width + rows)
    move = _unaligned if off else (lambda t: t)
    x, y, w = move(_rand(rows, width, g=g)), move(_rand(rows, width, g=g)), move(_rand(width, g=g))
    xd, yd, wd = x.double(), y.double(), w.double()
    rms = lambda v: torch.sqrt(v.square().mean(1, keepdim=True) + 1e-5)
    for dtype in (torch.bfloat16, torch.float32):
        coef = (0.5, -0.25, 0.75, 0.125)
        parts = [c * yd ** (i + 1) / rms(yd ** (i + 1)) for i, c in enumerate(coef[:3])]
        _close(seqops.polynorm(y, coef, 1e-5, dtype), sum(parts) + coef[3], sum(p.abs() for p in parts) + coef[3], width)
        got = move(x.clone())
        xt = seqops.add_scalar_norm(got, y, 0.7, 1e-5, dtype)
        ref, size = xd + 0.7 * yd / rms(yd), xd.abs() + (0.7 * yd / rms(yd)).abs()
        _close(got, ref, size, width)
        _close(xt, ref, size, width)
        got = move(x.clone())
        h = seqops.add_rms_norm(got, y, 1e-5, next_weight=w, dtype=dtype, around_zero=True)
        assert torch.equal(got, x + y)
        n = got.double() / rms(got.double())
        _close(h, n * (wd + 1), n.abs() * (wd.abs() + 1), width)
    got = x.clone()
    seqops.add_rms_norm(got, y, 1e-5)
    assert torch.equal(got, x + y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", [4, 6, 1020, 1028])
def test_embed_and_token_shift(width, dtype):
    from zhilight_amd import seqops
    lens = (1, 3, 2, 66)
    b, g = _batch(lens), torch.Generator(device=DEV).manual_seed(width)
    T = sum(lens)
    table, pos = _rand(50, width, g=g).to(dtype), _rand(60, width, g=g).to(dtype)
    tok = torch.randint(0, 50, (T,), device=DEV, dtype=torch.int32, generator=g)
    at = torch.cat([torch.arange(n) for n in lens]).clamp(max=59).to(DEV)
    assert torch.equal(seqops.embed(tok, table, None, 0.5, b), table[tok.long()].float() * 0.5)
    assert torch.equal(seqops.embed(tok, table, pos, 0.5, b), table[tok.long()].float() * 0.5 + pos[at].float())
    x, mix, prev = _rand(T, width, g=g), _rand(width, g=g), _rand(5, width, g=g)
    before, want_prev, start = torch.empty_like(x), prev.clone(), 0
    for i, n in enumerate(lens):
        before[start], before[start + 1:start + n] = prev[4 - i], x[start:start + n - 1]
        want_prev[4 - i] = x[start + n - 1]
        start += n
    ref = x.double() + (before.double() - x.double()) * mix.double()
    _close(seqops.token_shift(x, mix, prev, b, dtype), ref, x.double().abs() + ((before - x) * mix).double().abs(), 4)
    assert torch.equal(prev, want_prev)


# portions shorter than the taps, across and inside blocks of tokens, and blocks of one and of several tokens
@pytest.mark.parametrize("lens", [(1,), (1,) * 9, (2, 3, 1, 4, 5), (7, 2, 2, 1, 30), (8, 8, 16, 1), (2048, 1, 2, 3, 700, 5)])
@pytest.mark.parametrize("taps, channels", [(1, 8), (2, 1028), (3, 64), (4, 2052), (4, 30), (5, 8)])
def test_short_conv(taps, channels, lens):
    from zhilight_amd import seqops
    g = torch.Generator(device=DEV).manual_seed(taps + channels + len(lens))
    b, T, K = _batch(lens), sum(lens), taps - 1
    proj, w, bias, in_bias = _rand(T, channels + 8, g=g), _rand(channels, taps, g=g), _rand(channels, g=g), _rand(channels, g=g)
    tail = _rand(len(lens) + 1, K, channels, g=g)
    for col0, act in ((4, True), (8, False), (3, True)):
        got_tail = tail.clone() if K else None
        out, out_t = seqops.short_conv(proj, col0, w, in_bias, got_tail, b, act=act, bias=bias, also=torch.bfloat16)
        start, ref, size, want = 0, [], [], tail.clone()
        for i, n in enumerate(lens):
            seq = torch.cat([tail[len(lens) - i], proj[start:start + n, col0:col0 + channels] + in_bias])
            want[len(lens) - i] = seq[n:]
            win = seq.double().unfold(0, taps, 1) * w.double()
            ref.append(win.sum(2) + bias.double())
            size.append(win.abs().sum(2) + bias.double().abs())
            start += n
        ref, size = torch.cat(ref), torch.cat(size)
        if act:                                                                   # (SiLU's slope is below 1.1)
            ref, size = ref * torch.sigmoid(ref), 1.1 * size
        _close(out, ref, size, 4)
        _close(out_t, ref, size, 4)
        if K:
            assert torch.equal(got_tail, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, vdim, groups", [(2, 16, 2), (4, 64, 4), (3, 128, 3), (2, 256, 2), (4, 128, 2), (2, 48, 2), (2, 128, 1), (1, 4, 1), (5, 512, 5),
                                                 (2, 2050, 2), (1, 4096, 1), (1, 4100, 1)])
def test_group_norms(heads, vdim, groups, dtype):
    from zhilight_amd import seqops
    inner, g = heads * vdim, torch.Generator(device=DEV).manual_seed(heads + vdim)
    for rows in (1, 19):
        y, proj, w = _rand(rows, inner, g=g), _rand(rows, inner + 8, g=g), _rand(inner, g=g)
        for col0 in (4, 6):
            z = proj[:, col0:col0 + inner].double()
            v = y.double() * torch.nn.functional.silu(z)
            v = v.view(rows, groups, -1)
            ref = (v / torch.sqrt(v.square().mean(2, keepdim=True) + 1e-5)).view(rows, inner) * w.double()
            _close(seqops.gated_group_norm(y, proj, col0, w, 1e-5, groups, dtype), ref, ref.abs(), inner // groups)
            v = (y.double() * 0.3).view(rows, groups, -1)
            n = (v / torch.sqrt(v.square().mean(2, keepdim=True) + 1e-5)).view(rows, inner) * 0.5
            for act, f in (("silu", torch.nn.functional.silu), ("sigmoid", torch.sigmoid)):
                ref = n * w.double() * f(z)
                _close(seqops.linear_attn_finish(y, False, 0.3, None, 0.0, heads, vdim, groups, w, 1e-5, proj, col0, dtype, gate_act=act, out_scale=0.5),
                       ref, ref.abs(), inner // groups)
            _close(seqops.linear_attn_finish(y, False, 0.3, None, 0.0, heads, vdim, groups, None, 1e-5, None, 0, dtype, out_scale=0.5), n, n.abs(),
                   inner // groups)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, kv_heads, vdim", [(1, 1, 4), (4, 2, 6), (8, 2, 64), (16, 4, 128), (5, 5, 52)])
def test_plain_heads_gate(heads, kv_heads, vdim, dtype):
    from zhilight_amd import seqops
    lens = (1, 5, 13)
    b, T, width = _batch(lens), sum(lens), heads * vdim
    g = torch.Generator(device=DEV).manual_seed(heads + vdim)
    acc, sink = _rand(T, heads, 1, vdim, g=g), _rand(heads, g=g)
    ml = torch.stack([_rand(T, heads, 1, g=g), torch.rand(T, heads, 1, device=DEV, generator=g) + 0.1], 3).contiguous()
    gate = _rand(T, width + 8, g=g)
    m, l = ml[..., 0, 0].double(), ml[..., 0, 1].double()
    for sk, plain in ((None, False), (sink, False), (None, True)):
        f = torch.ones_like(l) if plain else 1 / l if sk is None else 1 / (l + torch.exp(sk.double() - m))
        for kind, col0 in ((None, 0), ("head", 3), ("full", 4), ("full", 5)):
            gt = None if kind is None else gate[:, col0:col0 + (heads if kind == "head" else width)].double().sigmoid()
            gt = 1.0 if gt is None else gt.view(T, heads, -1)
            ref = (acc[:, :, 0].double() * f[..., None] * gt * 0.5).reshape(T, width)
            out = seqops.head_mix_gate(acc, ml, 1, None, None, None if kind is None else gate, col0, b, heads, kv_heads, vdim, dtype, sink=sk,
                                       plain_sum=plain, gate_per_head=kind == "head", out_scale=0.5)
            _close(out, ref, ref.abs(), 256)


@pytest.mark.parametrize("bshd", [True, False])
@pytest.mark.parametrize("tasks, len_q, hkv, d", [(1, 1, 1, 8), (3, 1, 8, 128), (1, 300, 36, 64), (2, 77, 3, 24), (1, 5, 40, 512), (2, 130, 1, 8)])
def test_kv_scatter(tasks, len_q, hkv, d, bshd):
    """whole numbers: every placed row where it belongs, slots below 0 and past the buffer never written"""
    from zhilight_amd import ops
    g = torch.Generator(device=DEV).manual_seed(len_q + d)
    k, v = (torch.randint(-9, 9, (tasks, len_q, hkv, d), device=DEV, generator=g).half() for _ in range(2))
    lens = torch.tensor([len_q + 3 + i for i in range(tasks)], dtype=torch.int32, device=DEV)
    place = torch.stack([torch.randperm(len_q + 5, device=DEV, generator=g)[:len_q] - 1 for _ in range(tasks)]).int()      # -1 .. len_q + 3
    bufs = [[torch.full((n, hkv, d) if bshd else (hkv, n, d), 77.0, dtype=torch.float16, device=DEV) for n in lens.tolist()] for _ in range(2)]
    want = [[x.clone() for x in side] for side in bufs]
    for side, src in zip(want, (k, v)):
        for b in range(tasks):
            for t, p in enumerate(place[b].tolist()):
                if 0 <= p < int(lens[b]):
                    if bshd:
                        side[b][p] = src[b, t]
                    else:
                        side[b][:, p] = src[b, t]
    addr = [torch.tensor([x.data_ptr() for x in side], dtype=torch.int64, device=DEV) for side in bufs]
    ops.copy_to_rag_buffer2(place.contiguous(), lens, k, v, *addr, bshd=bshd)
    for side, ref in zip(bufs, want):
        assert all(torch.equal(a, r) for a, r in zip(side, ref))
