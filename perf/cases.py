"""Performance cases of the serving paths: what a program that serves models with this package has it do.

Llama-family models (zhilight_amd.llama.LLaMA, the geometries that ModelConfig names), in the three weight formats served in earnest:
  * "decode": one greedy step of a batch behind key / value histories -- the batch state is uploaded (one copy) and the captured step
    replayed, which is how a scheduler drives decoding.  Returned: logits and the key / value rows that the step wrote.
  * "prompt": `LLaMA.prefill` of one task's prompt, whole or in chunks.  Returned: the last row's logits and the prompt's keys and values.
Models on the ragged-step engine (zhilight_amd.engine.Engine.run_step; the widths of bench.py's "1b" and "8b" stacks, four layers):
  * "ragged": prompts of several requests of unequal lengths in one step, then `steps` single-token steps of all of them, then release.
    Returned: every step's logits (which depend on all that the caches and states hold).

Weights are drawn on the GPU in the checkpoint's own format and taken through the loaders; `exact` evaluates the same checkpoint in float64
with plain torch.  Depth is 8 layers of the real width (all 32 in the headline step): layers repeat, and a state has to be made quickly.  INT8
stacks have 4: a rounding to 8 bits turns a last-bit difference of its input into a whole code now and then, and depth piles these up.
"""
import math

import torch

DEV = "cuda:0"
F64 = torch.float64
GROUP = 128

LLAMA = {  # dim, heads, kv heads, head size, ff, vocabulary, rotary base, epsilon, and MiniCPM's scalings (embedding, depth, logits)
    "llama3_8b": dict(dim=4096, heads=32, kv=8, d=128, ff=14336, vocab=128256, theta=500000.0, eps=1e-5, emb=1.0, depth=0.0, base=0),
    "minicpm_2b": dict(dim=2304, heads=36, kv=36, d=64, ff=5760, vocab=122753, theta=10000.0, eps=1e-5, emb=12.0, depth=1.4, base=256),
}
RAGGED = {  # bench.py's stacks
    "1b": dict(width=2048, heads=16, kv_heads=4, dim=128, rank=512, ff2=8192, ff3=5440, m_heads=64, m_vdim=64, state=128, groups=8, window=1024,
               keep=8, taps=4, rot=64, low=16),
    "8b": dict(width=4096, heads=32, kv_heads=8, dim=128, rank=512, ff2=21504, ff3=9536, m_heads=128, m_vdim=64, state=128, groups=8, window=1024,
               keep=8, taps=4, rot=64, low=16),
}
RAGGED_VOCAB = 32000


def listed():
    return [
        # the smallest latency that a user sees: one sequence, a 1k history, the whole 32-layer model (the repository's headline workload)
        dict(name="w4 decode 1", kind="decode", model="llama3_8b", weights="w4", layers=32, batch=1, context=1024, ragged=False),
        # a full continuous batch: 32 sequences of unequal lengths
        dict(name="w4 decode 32 ragged", kind="decode", model="llama3_8b", weights="w4", layers=8, batch=32, context=1024, ragged=True),
        # a half-full INT8 server behind longer histories
        dict(name="int8 decode 8", kind="decode", model="llama3_8b", weights="int8", layers=4, batch=8, context=2000, ragged=False),
        # a few chats with a small unquantised model
        dict(name="bf16 decode 4", kind="decode", model="minicpm_2b", weights="bf16", layers=8, batch=4, context=300, ragged=True),
        # a one-line question
        dict(name="w4 prompt 57", kind="prompt", model="llama3_8b", weights="w4", layers=8, tokens=57, chunk=0),
        # time to first token of the benchmark's prompt
        dict(name="w4 prompt 1024", kind="prompt", model="llama3_8b", weights="w4", layers=8, tokens=1024, chunk=0),
        # a long document in pieces, as a scheduler that keeps decoding in between feeds it
        dict(name="w4 prompt 4096 in 1024", kind="prompt", model="llama3_8b", weights="w4", layers=8, tokens=4096, chunk=1024),
        # a document for the INT8 server, of no round length
        dict(name="int8 prompt 1000", kind="prompt", model="llama3_8b", weights="int8", layers=4, tokens=1000, chunk=0),
        # a page of text for the small model (64-wide heads, one kv head per head)
        dict(name="bf16 prompt 777", kind="prompt", model="minicpm_2b", weights="bf16", layers=8, tokens=777, chunk=0),
        # latent attention and state-space layers: one long prompt
        dict(name="latent+ssm 1b prompt 2048", kind="ragged", model="tupitar", size="1b", requests=1, tokens=2048, steps=0),
        # the same design, large: eight short requests come in together and are answered token by token
        dict(name="latent+ssm 8b chat 8", kind="ragged", model="tupitar", size="8b", requests=8, tokens=90, steps=12),
        # windowed grouped attention and gated linear attention: three unequal prompts in one step
        dict(name="window+gla 1b prompts", kind="ragged", model="gutivik", size="1b", requests=3, tokens=1300, steps=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "ragged"])
    if kind == "ragged":
        model, size, steps = rng.choice(["tupitar", "gutivik"]), rng.choice(["1b", "8b"]), rng.choice([0, 0, rng.randint(1, 12)])
        requests = rng.randint(1, 8)
        return dict(kind=kind, model=model, size=size, requests=requests, tokens=_log(rng, 20, min(2048, 4096 // requests)), steps=steps)
    weights = rng.choice(["w4", "w4", "int8", "bf16"])
    model = "minicpm_2b" if weights == "bf16" else "llama3_8b"
    layers = rng.choice([2, 4]) if weights == "int8" else rng.choice([2, 4, 8])
    if kind == "decode":
        return dict(kind=kind, model=model, weights=weights, layers=layers, batch=_log(rng, 1, 32), context=_log(rng, 100, 3000), ragged=rng.random() < 0.5)
    tokens = _log(rng, 16, 1024 if weights == "bf16" else 4096)
    chunk = rng.choice([0, 0, 512, 1024])
    return dict(kind=kind, model=model, weights=weights, layers=layers, tokens=tokens, chunk=chunk if chunk < tokens else 0)


# ---- checkpoints -------------------------------------------------------------------------------------------------------------------
def _gen(seed, what=0):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1000 + what)


def _randn(g, *shape, s=1.0, dtype=torch.float32):
    return torch.randn(shape, generator=g, device=DEV).mul_(s).to(dtype)


def _linears(z):
    hd, kvd = z["heads"] * z["d"], z["kv"] * z["d"]
    return [("attn.project_q", z["dim"], hd), ("attn.project_k", z["dim"], kvd), ("attn.project_v", z["dim"], kvd), ("attn.attn_out", hd, z["dim"]),
            ("ff.w_in", z["dim"], z["ff"]), ("ff.w_gated", z["dim"], z["ff"]), ("ff.w_out", z["ff"], z["dim"])]


def _llama_layer(case, z, seed, i):
    """One layer's checkpoint tensors.  w4: GPTQ words of uniform nibbles, stored zeros 0..14, half-normal scales; otherwise normal rows."""
    g, dt = _gen(seed, 10 + i), torch.bfloat16 if case["weights"] == "bf16" else torch.float16
    p = "llama.layers.%d." % i
    sd = {p + n + ".weight": (1 + _randn(g, z["dim"], s=0.1)).to(dt) for n in ("ln_attn", "ln_ff")}
    for name, k, n in _linears(z):
        if case["weights"] == "w4":
            sd[p + name + ".qweight"] = torch.randint(-2 ** 31, 2 ** 31, (k // 8, n), generator=g, device=DEV, dtype=torch.int32)
            nib = torch.randint(0, 15, (k // GROUP, n // 8, 8), generator=g, device=DEV, dtype=torch.int32)
            sd[p + name + ".qzeros"] = (nib << (4 * torch.arange(8, device=DEV, dtype=torch.int32))).sum(-1, dtype=torch.int32)
            sd[p + name + ".scales"] = (_randn(g, k // GROUP, n).abs() * (0.125 / math.sqrt(k)) + 1e-4).half()
        else:
            sd[p + name + ".weight"] = _randn(g, n, k, s=0.7 * k ** -0.5, dtype=dt)
    return sd


def _llama_ends(case, z, seed):
    g, dt = _gen(seed, 1), torch.bfloat16 if case["weights"] == "bf16" else torch.float16
    sd = {"llama.token_embedding.weight": _randn(g, z["vocab"], z["dim"], s=0.5 / z["emb"], dtype=dt),
          "llama.output_layernorm.weight": (1 + _randn(g, z["dim"], s=0.1)).to(dt)}
    if not z["base"]:                                                           # (MiniCPM's projection is its embedding)
        sd["llama.lm_head.weight"] = _randn(g, z["vocab"], z["dim"], s=0.02, dtype=dt)
    return sd


def _contexts(case):
    """The histories' lengths of a decode batch."""
    c, b = case["context"], case["batch"]
    return [max(1, c - (i * 37 * c // 100) % (c // 2 + 1)) if case["ragged"] else c for i in range(b)]


def _decode_inputs(case, z, seed):
    g, dt = _gen(seed, 2), torch.bfloat16 if case["weights"] == "bf16" else torch.float16
    tokens = torch.randint(0, z["vocab"], (case["batch"],), generator=g, device=DEV, dtype=torch.int32)
    kv = [_randn(g, case["layers"], 2, n, z["kv"], z["d"], dtype=dt) for n in _contexts(case)]
    return tokens, kv


def _prompt_tokens(case, z, seed):
    return torch.randint(0, z["vocab"], (case["tokens"],), generator=_gen(seed, 2), device=DEV, dtype=torch.int32)


def _lengths(case):
    n = case["tokens"]
    return [max(1, n - (i * 41 * n // 100) % (n // 2 + 1)) for i in range(case["requests"])]


def _ragged_tokens(case, seed):
    """Per request: its prompt and the tokens fed after it."""
    g = torch.Generator().manual_seed(int(seed) * 7 + 3)
    return [torch.randint(0, RAGGED_VOCAB, (n + case["steps"],), generator=g).tolist() for n in _lengths(case)]


def _ragged_config(case):
    z = RAGGED[case["size"]]
    if case["model"] == "tupitar":
        ff = dict(ff=z["ff2"], kind="dense")
        att = dict(type="latent_attention", mixer=dict(heads=z["heads"], dim=z["dim"], vdim=z["dim"], kv_rank=z["rank"], scale=z["dim"] ** -0.5), mlp=ff)
        ssm = dict(type="mamba2", mixer=dict(heads=z["m_heads"], vdim=z["m_vdim"], state=z["state"], groups=z["groups"], conv=4, norm_groups=z["groups"]), mlp=ff)
        return dict(architecture="Tupitar", vocab=RAGGED_VOCAB, width=z["width"], max_positions=2112, embedding=dict(scale=4.0), norm=dict(eps=1e-6),
                    layers=[att, att, ssm, att])
    ff = dict(ff=z["ff3"], kind="dense")
    att = dict(type="attention", mlp=ff, mixer=dict(heads=z["heads"], kv_heads=z["kv_heads"], dim=z["dim"], vdim=z["dim"], scale=z["dim"] ** -0.5, conv=z["taps"],
                                                    mask=dict(size=z["window"], keep_first=z["keep"]), rot=dict(dims=z["rot"], base=1e6), v_mix=True))
    gla = dict(type="gla", mlp=ff, mixer=dict(heads=z["heads"], dim=z["dim"], vdim=z["dim"], tau=16.0))
    return dict(architecture="Gutivik", vocab=RAGGED_VOCAB, width=z["width"], norm=dict(eps=1e-6), logit_scale=0.5, logit_softcap=20.0,
                layers=[att, gla, gla, att])


def _ragged_weights(case, seed):
    """Checkpoint of the configuration in bf16, one tensor after the other from one generator."""
    cfg, z, g = _ragged_config(case), RAGGED[case["size"]], _gen(seed, 5)
    W = cfg["width"]

    def rn(*shape, s=1.0, at=0.0):
        return (at + _randn(g, *shape, s=s)).to(torch.bfloat16)
    sd = {"embed": rn(RAGGED_VOCAB, W, s=0.25 if case["model"] == "tupitar" else 1.0), "head": rn(RAGGED_VOCAB, W, s=W ** -0.5)}
    if case["model"] == "tupitar":
        sd["pos"], sd["final.norm"] = rn(cfg["max_positions"], W, s=0.3), rn(s=0.1, at=1.0)
    else:
        sd["final.norm"] = rn(W, s=0.1)
    for i, layer in enumerate(cfg["layers"]):
        p, m, kind, ff = "l%d." % i, layer["mixer"], layer["type"], layer["mlp"]["ff"]
        H, D, V = m["heads"], m.get("dim", 0), m["vdim"]
        if kind == "mamba2":
            inner, gn = H * V, m["groups"] * m["state"]
            sd.update({p + "mix.in": rn(2 * inner + 2 * gn + H, W, s=W ** -0.5), p + "mix.conv": rn(inner + 2 * gn, 4, s=0.5), p + "mix.conv.b": rn(inner + 2 * gn, s=0.2),
                       p + "mix.dt_bias": rn(H), p + "mix.A_log": rn(H, s=0.8, at=-1.5), p + "mix.D": rn(H), p + "mix.norm": rn(inner, s=0.2, at=1.0)})
        elif kind == "latent_attention":
            r = m["kv_rank"]
            sd.update({p + "mix.q": rn(H * D, W, s=W ** -0.5), p + "mix.dkv": rn(r, W, s=W ** -0.5), p + "mix.dkv.norm": rn(r, s=0.2, at=1.0),
                       p + "mix.uk": rn(H * D, r, s=r ** -0.5), p + "mix.uv": rn(H * V, r, s=r ** -0.5), p + "mix.sink": rn(H), p + "mix.g": rn(H, W, s=W ** -0.5)})
        elif kind == "attention":
            for n, rows in (("q", H * D), ("k", m["kv_heads"] * D), ("v", m["kv_heads"] * V)):
                sd.update({p + "mix." + n: rn(rows, W, s=W ** -0.5), p + "mix.%s.b" % n: rn(rows, s=0.1), p + "mix.%s.conv" % n: rn(rows, m["conv"], s=m["conv"] ** -0.5)})
            sd.update({p + "mix.sink": rn(H), p + "mix.vmix": torch.tensor([0.375], dtype=torch.bfloat16, device=DEV)})
        else:
            sd.update({p + "mix." + n: rn(H * D, W, s=W ** -0.5) for n in ("q", "k", "v", "g")})
            sd.update({p + "mix.a1": rn(z["low"], W, s=W ** -0.5), p + "mix.a2": rn(H * D, z["low"], s=z["low"] ** -0.5), p + "mix.a2.b": rn(H * D, s=0.5, at=2.0),
                       p + "mix.norm": rn(V, s=0.2, at=1.0)})
        sd[p + "mix.o"] = rn(W, H * V, s=(H * V) ** -0.5)
        if case["model"] == "tupitar":
            sd.update({p + "norm1": rn(s=0.1, at=1.0), p + "norm2": rn(s=0.1, at=1.0), p + "shift": torch.rand(W, generator=g, device=DEV).to(torch.bfloat16),
                       p + "mlp.up": rn(ff, W, s=W ** -0.5), p + "mlp.act": torch.tensor([1.0, 0.25, 0.125, 0.125], dtype=torch.bfloat16, device=DEV)})
        else:
            sd.update({p + "norm1": rn(W, s=0.1), p + "norm2": rn(W, s=0.1), p + "mlp.gate": rn(ff, W, s=W ** -0.5), p + "mlp.up": rn(ff, W, s=W ** -0.5)})
        sd[p + "mlp.down"] = rn(W, ff, s=ff ** -0.5)
    return cfg, sd


# ---- what a program holds before the call -------------------------------------------------------------------------------------------
def _load_llama(case, seed):
    from zhilight_amd.llama import LLaMA, ModelConfig, QuantConfig
    z = LLAMA[case["model"]]
    cfg = ModelConfig.llama3_8b() if case["model"] == "llama3_8b" else ModelConfig.minicpm_2b()
    cfg.num_layers = case["layers"]
    model = LLaMA(cfg, {"w4": QuantConfig(5, GROUP), "int8": QuantConfig(2, 0), "bf16": QuantConfig(0)}[case["weights"]], DEV)
    sd = _llama_ends(case, z, seed)
    for i in range(case["layers"]):
        sd.update(_llama_layer(case, z, seed, i))
    return model.load_state_dict(sd, hf_names=False), z


def prepare(case, seed):
    if case["kind"] == "ragged":
        from zhilight_amd.engine import Engine, Entry
        from zhilight_amd.registry import model_class
        cfg, sd = _ragged_weights(case, seed)
        model = model_class(cfg).from_config(cfg, dtype="bfloat16", device=DEV).load_weights(sd)
        toks, lens = _ragged_tokens(case, seed), _lengths(case)
        names = ["r%d" % i for i in range(case["requests"])]
        steps = [[Entry(r, t[:n], [n - 1]) for r, t, n in zip(names, toks, lens)]]
        steps += [[Entry(r, [t[n + s]], [0]) for r, t, n in zip(names, toks, lens)] for s in range(case["steps"])]
        eng = Engine(model, max_tokens=sum((n + case["steps"] + 63) // 64 * 64 for n in lens), max_seqs=len(names))
        return dict(case=case, engine=eng, steps=steps, names=names)
    model, z = _load_llama(case, seed)
    if case["kind"] == "prompt":
        n = case["tokens"]
        ctx = model.new_context(1, (n + 64) // 64 * 64 + 64, 0)
        return dict(case=case, model=model, ctx=ctx, prompt=_prompt_tokens(case, z, seed), written=ctx.kv[0][:, :, :n])
    tokens, history = _decode_inputs(case, z, seed)
    lens = _contexts(case)
    ctx = model.new_context(len(lens), (max(lens) + 64) // 64 * 64 + 64, max(lens))
    for t, h in zip(ctx.kv, history):
        t[:, :, :h.shape[2]] = h
    pos = torch.tensor(lens, dtype=torch.int32, device=DEV)
    start = torch.stack([tokens, pos, pos, pos + 1])
    live = start.clone()
    ctx.tokens, ctx.positions, ctx.placement, ctx.valid_lens = live.unbind(0)
    ctx.steps_left = 1 << 60                                                    # (the same step every time: the buffers never fill)

    def step():
        live.copy_(start)
        return model.step_greedy(ctx)[0]
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = step()
    return dict(case=case, graph=graph, keep=(model, ctx, live, start), out=[logits, [t[:, :, n] for t, n in zip(ctx.kv, lens)]])


def run(state):
    kind = state["case"]["kind"]
    if kind == "decode":
        state["graph"].replay()
        return state["out"]
    if kind == "prompt":
        return [state["model"].prefill(state["ctx"], 0, state["prompt"], state["case"]["chunk"]), state["written"]]
    eng = state["engine"]
    out = [eng.run_step(entries) for entries in state["steps"]]
    for r in state["names"]:
        eng.release(r)
    return out


# ---- what a pass cannot do without --------------------------------------------------------------------------------------------------
def work(case):
    if case["kind"] == "ragged":
        z, lens, steps = RAGGED[case["size"]], _lengths(case), case["steps"]
        W, H, D = z["width"], z["heads"], z["dim"]
        if case["model"] == "tupitar":
            ff, inner = 2 * W * z["ff2"], z["m_heads"] * z["m_vdim"]
            att = (H * D + z["rank"] + H) * W + W * H * D + ff
            ssm = (2 * inner + 2 * z["groups"] * z["state"] + z["m_heads"]) * W + W * inner + ff
            mats, up = 3 * att + ssm, 3 * 2 * H * D * z["rank"]                # up: the keys and values of every cached latent
            pair, walk, rows = 3 * 4 * H * D, 6 * inner * z["state"], 3 * z["rank"] * 2
            state = inner * z["state"] * 4 * 2
        else:
            ff, kvd = 3 * W * z["ff3"], z["kv_heads"] * D
            mats, up = 2 * ((H * D + 2 * kvd) * W + W * H * D + ff) + 2 * (4 * H * D * W + z["low"] * (W + H * D) + W * H * D + ff), 0
            pair, walk, rows = 2 * 4 * H * D, 2 * 5 * H * D * D, 2 * 2 * kvd * 2
            state = 2 * H * D * D * 4 * 2
        window = z["window"] + z["keep"] if case["model"] == "gutivik" else 1 << 30
        n = sum(lens)
        pairs = sum(min(t + 1, window) for k in lens for t in range(k + steps))
        read = sum(min(k + s, window) for k in lens for s in range(steps))      # cached rows that the single tokens look back at
        flops = 2 * (n + steps * len(lens)) * (mats + up) + 2 * (1 + steps) * len(lens) * RAGGED_VOCAB * W + pairs * pair + (n + steps * len(lens)) * walk
        nbytes = (1 + steps) * 2 * (mats + up + RAGGED_VOCAB * W) + (n + read) * rows + (1 + steps) * len(lens) * (state + RAGGED_VOCAB * 4)
        return {"bytes": nbytes, "flops": flops}
    z = LLAMA[case["model"]]
    par = sum(k * n for _, k, n in _linears(z)) * case["layers"]
    wb = par * {"w4": 0.5 + 2.5 / GROUP, "int8": 1.0, "bf16": 2.0}[case["weights"]]
    row = 2 * 2 * z["kv"] * z["d"] * case["layers"]                             # key and value bytes of one token
    head = z["vocab"] * z["dim"]
    if case["kind"] == "decode":
        lens = _contexts(case)
        return {"bytes": wb + 2 * head + row * (sum(lens) + len(lens)) + 2 * z["vocab"] * len(lens),
                "flops": 2 * len(lens) * (par + head) + 4 * z["heads"] * z["d"] * case["layers"] * (sum(lens) + len(lens))}
    n = case["tokens"]
    return {"bytes": wb + 2 * head + row * n + 2 * z["dim"] * n + 2 * z["vocab"],
            "flops": 2 * n * par + 2 * head + 4 * z["heads"] * z["d"] * case["layers"] * n * (n + 1) // 2}


def tolerance(case):
    # 16-bit activations between the layers: about four times what the path is from its float64 evaluation (fp16 rows 6e-4 .. 5e-3 at depth 8,
    # bf16 5e-3 .. 8e-3; the INT8 stack, whose activations are rounded to 8 bits, 1.4e-2 .. 2.3e-2, and there no more than this can be allowed)
    if case["kind"] == "ragged":
        return {"rel": 0.02 if case["model"] == "tupitar" else 0.03, "max": 0.3}
    return {"w4": {"rel": 0.015, "max": 0.3}, "int8": {"rel": 0.03, "max": 0.4}, "bf16": {"rel": 0.03, "max": 0.4}}[case["weights"]]


# ---- the same in float64 ------------------------------------------------------------------------------------------------------------
def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _dequantised(sd, name):
    """(K, N) float64 of a GPTQ linear."""
    q, zr, s = sd[name + ".qweight"], sd[name + ".qzeros"], sd[name + ".scales"]
    shift = 4 * torch.arange(8, device=DEV, dtype=torch.int32)
    k, n = q.shape[0] * 8, q.shape[1]
    nib = ((q[:, None, :] >> shift[None, :, None]) & 15).reshape(k // GROUP, GROUP, n).to(F64)
    zero = ((zr[:, :, None] >> shift) & 15).reshape(k // GROUP, 1, n).to(F64) + 1
    return ((nib - zero) * s.to(F64)[:, None, :]).reshape(k, n)


def _codes(x):
    """Rows as whole numbers of their largest magnitude's 127th."""
    s = x.abs().amax(-1, keepdim=True) / 127
    return torch.round(x / s), s


def _linear64(case, sd, name):
    if case["weights"] == "w4":
        w = _dequantised(sd, name)
        return lambda x: x @ w
    w = sd[name + ".weight"].to(F64)
    if case["weights"] == "bf16":
        return lambda x: x @ w.T
    wq, ws = _codes(w)
    ws = ws.half().to(F64)

    def f(x):
        xq, xs = _codes(x)
        return (xq @ wq.T) * xs * ws.T
    return f


def _rope(x, pos, theta):
    """x (T, heads, d): halves paired."""
    d = x.shape[-1]
    ang = pos.to(F64)[:, None] * theta ** (-torch.arange(0, d, 2, device=DEV, dtype=F64) / d)
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, k, v, scale, vis, sink=None):
    """q (T, H, d), k / v (S, G, d), vis (T, S)."""
    H, G = q.shape[1], k.shape[1]
    out = torch.empty(q.shape[0], H, v.shape[2], dtype=F64, device=DEV)
    for h in range(H):
        s = ((q[:, h] @ k[:, h * G // H].T) * scale).masked_fill_(~vis, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].expand(s.shape[0], 1)], 1)
        out[:, h] = torch.softmax(s, 1)[:, :k.shape[0]] @ v[:, h * G // H]
    return out


def _exact_llama(case, seed):
    z = LLAMA[case["model"]]
    ends = _llama_ends(case, z, seed)
    decode = case["kind"] == "decode"
    if decode:
        tokens, history = _decode_inputs(case, z, seed)
        pos = torch.tensor(_contexts(case), device=DEV)
    else:
        tokens = _prompt_tokens(case, z, seed)
        pos = torch.arange(case["tokens"], device=DEV)
        vis = pos[:, None] >= pos[None, :]
    x = ends["llama.token_embedding.weight"][tokens.long()].to(F64) * z["emb"]
    add = z["depth"] / math.sqrt(case["layers"]) if z["depth"] else 1.0
    H, G, d, rows = z["heads"], z["kv"], z["d"], []
    for i in range(case["layers"]):
        sd, p = _llama_layer(case, z, seed, i), "llama.layers.%d." % i
        h = _rms(x, sd[p + "ln_attn.weight"].to(F64), z["eps"])
        q, k, v = (_linear64(case, sd, p + "attn.project_" + n)(h).view(len(pos), -1, d) for n in "qkv")
        q, k = _rope(q, pos, z["theta"]), _rope(k, pos, z["theta"])
        if decode:
            past = [t[i].to(F64) for t in history]
            o = torch.cat([_attend(q[b:b + 1], torch.cat([past[b][0], k[b:b + 1]]), torch.cat([past[b][1], v[b:b + 1]]), d ** -0.5,
                                   torch.ones(1, past[b].shape[1] + 1, dtype=torch.bool, device=DEV)) for b in range(len(pos))])
        else:
            o = _attend(q, k, v, d ** -0.5, vis)
        rows.append(torch.stack([k, v]))
        x = x + add * _linear64(case, sd, p + "attn.attn_out")(o.reshape(len(pos), H * d))
        h = _rms(x, sd[p + "ln_ff.weight"].to(F64), z["eps"])
        a = torch.nn.functional.silu(_linear64(case, sd, p + "ff.w_in")(h)) * _linear64(case, sd, p + "ff.w_gated")(h)
        x = x + add * _linear64(case, sd, p + "ff.w_out")(a)
    x = x if decode else x[-1:]
    head = ends.get("llama.lm_head.weight", ends["llama.token_embedding.weight"])
    x = _rms(x, ends["llama.output_layernorm.weight"].to(F64), z["eps"]) * (z["base"] / z["dim"] if z["base"] else 1.0)
    logits = torch.cat([x @ part.to(F64).T for part in head.split(16384)], 1)
    kv = torch.stack(rows)                                                      # (layers, 2, T, G, d)
    return [logits, list(kv.unbind(2)) if decode else kv]


def _conv(u, w, b):
    taps = w.shape[1]
    pad = torch.cat([u.new_zeros(taps - 1, u.shape[1]), u])
    return b + sum(pad[k:k + u.shape[0]] * w[:, k] for k in range(taps))


def _pairs_turned(x, pos, dims, base):
    ang = pos.to(F64)[:, None] * base ** (-torch.arange(0, dims, 2, device=DEV, dtype=F64) / dims)
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    u, v = x[..., 0:dims:2], x[..., 1:dims:2]
    out = x.clone()
    out[..., 0:dims:2], out[..., 1:dims:2] = u * c - v * s, v * c + u * s
    return out


def _tupitar_mixer(h, w, m, kind, eps):
    T, H, V = h.shape[0], m["heads"], m["vdim"]
    if kind == "latent_attention":
        c = _rms(h @ w("dkv").T, w("dkv.norm"), eps)
        t = torch.arange(T, device=DEV)
        o = _attend((h @ w("q").T).view(T, H, -1), (c @ w("uk").T).view(T, H, -1), (c @ w("uv").T).view(T, H, V), m["scale"], t[:, None] >= t[None, :], w("sink"))
        return (o * torch.sigmoid(h @ w("g").T)[:, :, None]).reshape(T, H * V) @ w("o").T
    N, G, R, inner = m["state"], m["groups"], m["norm_groups"], H * V
    zed, xbc, dt = (h @ w("in").T).split([inner, inner + 2 * G * N, H], 1)
    xbc = torch.nn.functional.silu(_conv(xbc, w("conv"), w("conv.b")))
    x = xbc[:, :inner].view(T, H, V)
    B, C = (xbc[:, inner + k * G * N:inner + (k + 1) * G * N].view(T, G, N).repeat_interleave(H // G, 1) for k in (0, 1))
    dt = torch.nn.functional.softplus(dt + w("dt_bias"), threshold=60.0)
    keep, dx = torch.exp(-torch.exp(w("A_log")) * dt), dt[:, :, None] * x
    S, y = h.new_zeros(H, N, V), torch.empty(T, H, V, dtype=F64, device=DEV)
    for t in range(T):
        S.mul_(keep[t][:, None, None]).addcmul_(B[t][:, :, None], dx[t][:, None, :])
        y[t] = (S * C[t][:, :, None]).sum(1)
    y = (y + w("D")[:, None] * x).reshape(T, inner) * torch.nn.functional.silu(zed)
    return (_rms(y.view(T, R, inner // R), 1.0, eps).reshape(T, inner) * w("norm")) @ w("o").T


def _tupitar64(cfg, sd, tokens):
    eps, T = cfg["norm"]["eps"], len(tokens)
    x = sd["embed"][torch.tensor(tokens, device=DEV)].to(F64) * cfg["embedding"]["scale"] + sd["pos"][:T].to(F64)
    for i, layer in enumerate(cfg["layers"]):
        def w(n, p="l%d." % i):
            return sd[p + n].to(F64)
        h = x + (torch.cat([torch.zeros_like(x[:1]), x[:-1]]) - x) * w("shift")
        x = x + _rms(_tupitar_mixer(h, lambda n: w("mix." + n), layer["mixer"], layer["type"], eps), w("norm1"), eps)
        u, (a, b, c, e) = x @ w("mlp.up").T, w("mlp.act")
        x = x + _rms((a * _rms(u, 1.0, eps) + b * _rms(u * u, 1.0, eps) + c * _rms(u ** 3, 1.0, eps) + e) @ w("mlp.down").T, w("norm2"), eps)
    return lambda at: _rms(x[at], sd["final.norm"].to(F64), eps) @ sd["head"].to(F64).T


def _gutivik64(cfg, sd, tokens):
    eps, T = cfg["norm"]["eps"], len(tokens)
    x, first = sd["embed"][torch.tensor(tokens, device=DEV)].to(F64), None
    t = torch.arange(T, device=DEV)
    for i, layer in enumerate(cfg["layers"]):
        def w(n, p="l%d." % i):
            return sd[p + n].to(F64)
        m = layer["mixer"]
        H, D, V, h = m["heads"], m["dim"], m["vdim"], _rms(x, 1 + w("norm1"), eps)
        if layer["type"] == "attention":
            q, k, v = (_conv(h @ w("mix." + n).T + w("mix.%s.b" % n), w("mix.%s.conv" % n), 0.0).view(T, -1, D) for n in "qkv")
            q, k = (_pairs_turned(u, t, m["rot"]["dims"], m["rot"]["base"]) for u in (q, k))
            first, own = (v, v) if first is None else (first, (1 - w("mix.vmix")) * v + w("mix.vmix") * first)
            back = t[:, None] - t[None, :]
            o = _attend(q, k, own, m["scale"], (back >= 0) & ((back < m["mask"]["size"]) | (t[None, :] < m["mask"]["keep_first"])), w("mix.sink")).reshape(T, H * V)
        else:
            q, k, v = ((h @ w("mix." + n).T).view(T, H, -1) for n in "qkv")
            keep = torch.exp(torch.nn.functional.logsigmoid(h @ w("mix.a1").T @ w("mix.a2").T + w("mix.a2.b")) / m["tau"]).view(T, H, D)
            S, o = x.new_zeros(H, D, V), torch.empty(T, H, V, dtype=F64, device=DEV)
            for s in range(T):
                S.mul_(keep[s][:, :, None]).addcmul_(k[s][:, :, None], v[s][:, None, :])
                o[s] = (S * q[s][:, :, None]).sum(1)
            o = _rms(o * D ** -0.5, w("mix.norm"), eps).reshape(T, H * V) * torch.nn.functional.silu(h @ w("mix.g").T)
        x = x + o @ w("mix.o").T
        h = _rms(x, 1 + w("norm2"), eps)
        x = x + (torch.nn.functional.gelu(h @ w("mlp.gate").T, approximate="tanh") * (h @ w("mlp.up").T)) @ w("mlp.down").T

    def logits(at):
        y = _rms(x[at], 1 + sd["final.norm"].to(F64), eps) @ sd["head"].to(F64).T * cfg["logit_scale"]
        return cfg["logit_softcap"] * torch.tanh(y / cfg["logit_softcap"])
    return logits


def exact(case, seed):
    if case["kind"] != "ragged":
        return _exact_llama(case, seed)
    cfg, sd = _ragged_weights(case, seed)
    model = _tupitar64 if case["model"] == "tupitar" else _gutivik64
    rows = [model(cfg, sd, toks)(torch.arange(n - 1, n + case["steps"], device=DEV)) for toks, n in zip(_ragged_tokens(case, seed), _lengths(case))]
    return list(torch.stack(rows, 1).unbind(0))
