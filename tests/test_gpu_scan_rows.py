"""The scan for states of whole 64s of rows (k_scan_rows in csrc_seq/ssm.hip) against a float64 walk over the tokens.

Bound: a state number is a sum of b x over the tokens, an output a sum of those over the rows; each step rounds at most three times (2^-24) and decays
are at most 1, so the error is below 4 (tokens + rows) 2^-24 times the same sums with absolute values."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _batch(lens):
    from zhilight_amd import seqops
    seqs, page = [], 0
    for i, n in enumerate(lens):
        k = (n + 63) // 64
        seqs.append((n, 0, len(lens) - i, list(range(page, page + k))))          # (slots in another order, slot 0 nobody's)
        page += k
    return seqops.RaggedBatch(seqs, 64, DEV)


def _walk(x, b, c, a, scale, state, lens):
    """x (T, H, P), b / c / a (T, H, N), scale (T, H), state (S, H, N, P) -> outputs, end states, and both with absolute values"""
    x, b, c, a, scale = (t.double() for t in (x, b, c, a, scale))
    y, yabs, S, at = torch.empty_like(x), torch.empty_like(x), state.double().clone(), 0
    Sabs = S.abs()
    for i, n in enumerate(lens):
        slot = len(lens) - i
        for t in range(at, at + n):
            add = b[t][:, :, None] * (scale[t][:, None] * x[t])[:, None, :]
            S[slot] = a[t][:, :, None] * S[slot] + add
            Sabs[slot] = a[t][:, :, None] * Sabs[slot] + add.abs()
            y[t], yabs[t] = (S[slot] * c[t][:, :, None]).sum(1), (Sabs[slot] * c[t].abs()[:, :, None]).sum(1)
        at += n
    return y, S, yabs, Sabs


def _close(got, ref, size, steps):
    assert bool(((got.double() - ref).abs() <= 4 * steps * 2.0 ** -24 * size + 1e-30).all())


# (rows, columns): the smallest, ragged waves, two chunk lengths (long rows are staged 8 tokens at a time), the largest
SIZES = [(64, 16), (64, 48), (128, 64), (128, 128), (128, 256), (256, 128), (64, 256)]


@pytest.mark.parametrize("kind", ["per channel", "per token", "per head"])
@pytest.mark.parametrize("N, P", SIZES)
def test_linear_attention_scan(N, P, kind):
    from zhilight_amd import seqops
    H = 2
    for lens, seg in (((1, 1), 0), ((7, 16, 17), 0), ((50, 3, 33), 16), ((40,), 24)):
        g = torch.Generator(device=DEV).manual_seed(N + P + sum(lens))
        T = sum(lens)
        proj = torch.randn(T, 4 + H * (2 * N + P), device=DEV, generator=g)
        state = torch.randn(len(lens) + 1, H, N, P, device=DEV, generator=g)
        act = kind == "per head"
        decay_h = torch.tensor([1.0, 0.9], device=DEV) if kind == "per head" else None
        decay_t = torch.rand(T, H, device=DEV, generator=g) if kind == "per token" else None
        gain = torch.rand(T, H, device=DEV, generator=g) if kind == "per token" else None
        decay_v = torch.rand(T, H * N, device=DEV, generator=g) if kind == "per channel" else None
        for d in (decay_t, decay_v):
            if d is not None:
                d[0], d[-1] = 0.0, 1.0
        q, k, v = (proj[:, s:s + H * w].reshape(T, H, w) for s, w in ((4, N), (4 + H * N, N), (4 + 2 * H * N, P)))
        if act:
            q, k, v = (t.double() * torch.sigmoid(t.double()) for t in (q, k, v))
        a = decay_v.view(T, H, N) if decay_v is not None else (decay_t if decay_t is not None else decay_h.expand(T, H))[:, :, None].expand(T, H, N)
        y, S, ya, Sa = _walk(v, k, q, a, gain if gain is not None else torch.ones(T, H, device=DEV), state, lens)
        got_state = state.clone()
        got = seqops.decay_scan(proj, 4, 4 + H * N, 4 + 2 * H * N, act, decay_h, decay_t, gain, False, got_state, H, N, P, _batch(lens), seg_len=seg, decay_v=decay_v)
        steps = max(lens) + N + (8 if act else 0)
        _close(got.view(T, H, P), y, ya, steps)
        _close(got_state, S, Sa, steps)
        assert torch.equal(got_state[0], state[0])


@pytest.mark.parametrize("N, P", SIZES)
def test_state_space_scan(N, P):
    """the Mamba-2 sources: step sizes through softplus, B and C shared by a group's heads, the skip term.  (The step size and the decay are fp32
    functions: a few ulp on top, multiplied up over the tokens that a number stays in the state.)"""
    from zhilight_amd import seqops
    H, G = 4, 2
    for lens, seg in (((1, 1, 1), 0), ((16, 9), 0), ((70, 20), 32)):
        g = torch.Generator(device=DEV).manual_seed(N + P + sum(lens))
        T = sum(lens)
        xbc = torch.randn(T, H * P + 2 * G * N, device=DEV, generator=g)
        proj = torch.randn(T, 8 + H, device=DEV, generator=g)
        bias, a_log, skip = (torch.randn(H, device=DEV, generator=g) for _ in range(3))
        state = torch.randn(len(lens) + 1, H, N, P, device=DEV, generator=g)
        x = xbc[:, :H * P].view(T, H, P)
        B, Cm = (xbc[:, H * P + i * G * N:H * P + (i + 1) * G * N].view(T, G, N).repeat_interleave(H // G, 1) for i in (0, 1))
        dt = torch.nn.functional.softplus(proj[:, 8:].double() + bias.double(), threshold=60.0)
        a = torch.exp(-torch.exp(a_log.double()) * dt)[:, :, None].expand(T, H, N)
        y, S, ya, Sa = _walk(x, B, Cm, a, dt, state, lens)
        y = y + skip.double()[None, :, None] * x.double()
        ya = ya + (skip[None, :, None] * x).abs().double()
        got_state = state.clone()
        got = seqops.ssm_scan(xbc, proj, 8, bias, a_log, skip, got_state, H, P, N, G, _batch(lens), seg_len=seg)
        steps = 12 * max(lens) + N
        _close(got.view(T, H, P), y, ya, steps)
        _close(got_state, S, Sa, steps)
