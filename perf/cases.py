"""The workloads whose speed this library is judged by: what a program that uses it has it do, through the public entry points.

`listed()` names twelve of them, `draw(rng)` gives more from the same ranges.  A case is a dict of plain values:

family   "neox", "llama" (fp16 operators, one token), "nibotar", "kagapel" (whole models, prompts and tokens)
path     neox: "layer" / "layer_split" (one decoder layer through the operator), "step" (one greedy step of a whole model);
         llama: "layer" (attention and MLP block), "plain" (the operator with [in, out] weights), "batch" (paged caches);
         models: "prompt" (a prompt from position 0), "turn" (more tokens of a sequence that has a context), "step" (one
         greedy step)
model    the sizes, by name
context  positions in the cache before the call (of every sequence on average with "batch")

Inputs have the scales that trained models have: matrices of standard deviation 0.02, those that write into the residual stream
of a model smaller with its depth (as deep models are made, so that a rounding in the first layer does not grow from layer to
layer), norm weights around one, hidden states and caches of order one."""
from __future__ import annotations

import math

import torch

DEV = "cuda:0"

NEOX = {
    "pythia_2b8": dict(hidden=2560, heads=32, head_dim=80, rotary_dim=20, ffn=10240, vocab=50304),
    "pythia_6b9": dict(hidden=4096, heads=32, head_dim=128, rotary_dim=32, ffn=16384, vocab=50432),
}
LLAMA = {"llama2_7b": dict(hidden=4096, heads=32, head_dim=128, ffn=11008, eps=1e-6)}
NIBOTAR = {
    "dense_6b9": dict(width=4096, heads=32, kv_heads=32, dim=128, vdim=128, chunk=8192, ff=16384, vocab=50432),
    "dense_8b": dict(width=4096, heads=32, kv_heads=8, dim=128, vdim=128, chunk=8192, ff=14336, vocab=128256),
    "experts_16b": dict(width=2048, heads=16, kv_heads=4, dim=128, vdim=128, chunk=8192, ff=1408, experts=64, top=6, shared=2816, vocab=102400),
    # small and uneven: rows that are no multiple of a tile, heads that are no multiple of 32 elements, short chunks
    "uneven": dict(width=1500, heads=12, kv_heads=4, dim=96, vdim=80, chunk=1000, ff=4100, vocab=32001),
}
KAGAPEL = {
    "latent_6b9": dict(width=4096, heads=32, dim=128, rot_dim=64, vdim=128, kv_rank=512, ff=11264, streams=4, vocab=50432),
    "latent_2b": dict(width=2048, heads=16, dim=128, rot_dim=64, vdim=128, kv_rank=512, ff=10944, streams=2, vocab=102400),
    "latent_wide": dict(width=5120, heads=128, dim=128, rot_dim=64, vdim=128, kv_rank=512, ff=12288, streams=4, vocab=102400),
    "uneven": dict(width=1500, heads=12, dim=72, rot_dim=32, vdim=88, kv_rank=200, ff=4100, streams=3, vocab=32001),
}
SEQ = {"nibotar": NIBOTAR, "kagapel": KAGAPEL}


def listed():
    return [
        # one layer of the smallest model inside somebody's own loop: the shortest call, where launch latency counts
        dict(name="neox_layer_2b8", family="neox", path="layer", model="pythia_2b8", context=511),
        # a token of the flagship model at the context that its speed is quoted for
        dict(name="neox_step_6b9", family="neox", path="step", model="pythia_6b9", layers=32, context=2048),
        # a LLaMA layer late in its context window
        dict(name="llama_layer", family="llama", path="layer", model="llama2_7b", context=4000),
        # a serving step: sixteen sequences of different lengths over paged caches
        dict(name="llama_batch_16", family="llama", path="batch", model="llama2_7b", batch=16, context=1024),
        # a long prompt of a dense model, as at the start of a conversation over a document
        dict(name="nibotar_prompt_6b9", family="nibotar", path="prompt", model="dense_6b9", dtype="bf16", layers=32, tokens=2048, context=0, want="last"),
        # a short message late in a conversation: few tokens, all of the weights
        dict(name="nibotar_turn_8b", family="nibotar", path="turn", model="dense_8b", dtype="bf16", layers=32, tokens=37, context=1990, want="last"),
        # a generated token of the same model
        dict(name="nibotar_step_8b", family="nibotar", path="step", model="dense_8b", dtype="bf16", layers=32, tokens=1, context=2048, want="last"),
        # an ordinary prompt of a model with many small experts
        dict(name="nibotar_prompt_experts", family="nibotar", path="prompt", model="experts_16b", dtype="bf16", layers=12, tokens=700, context=0, want="last"),
        # every logit of a prompt in float32: how a checkpoint is checked against another implementation (trace replay)
        dict(name="nibotar_score_f32", family="nibotar", path="prompt", model="uneven", dtype="f32", layers=8, tokens=301, context=0, want="all"),
        # the largest call: a document as long as the position vectors allow, latent attention
        dict(name="kagapel_prompt_6b9", family="kagapel", path="prompt", model="latent_6b9", dtype="bf16", layers=32, tokens=8000, context=0, want="last"),
        # a medium-sized message at some depth of a smaller latent-attention model
        dict(name="kagapel_turn_2b", family="kagapel", path="turn", model="latent_2b", dtype="bf16", layers=27, tokens=150, context=3001, want="last"),
        # a generated token with a long cache of latents
        dict(name="kagapel_step_6b9", family="kagapel", path="step", model="latent_6b9", dtype="bf16", layers=32, tokens=1, context=4096, want="last"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["neox", "llama", "nibotar", "nibotar", "kagapel", "kagapel"])
    if family == "neox":
        c = dict(family=family, path=rng.choice(["layer", "layer_split", "step"]), model=rng.choice(sorted(NEOX)), context=_log(rng, 1, 8192))
        if c["path"] == "step":
            c["layers"] = rng.randint(4, 32)
        return c
    if family == "llama":
        c = dict(family=family, path=rng.choice(["layer", "plain", "batch"]), model="llama2_7b", context=_log(rng, 16, 8192))
        if c["path"] == "batch":
            c.update(batch=_log(rng, 1, 64), context=_log(rng, 16, 2048))
        return c
    sizes = SEQ[family]
    path, model = rng.choice(["prompt", "turn", "step"]), rng.choice(sorted(sizes))
    c = dict(family=family, path=path, model=model, dtype="f32" if model == "uneven" and rng.random() < 0.5 else "bf16", layers=rng.randint(3, 12),
             tokens=1, context=0, want=rng.choice(["last", "last", "all"]) if path != "step" else "last")
    top = 4000
    if path == "prompt":
        c["tokens"] = _log(rng, 2, 8000 if c["want"] == "last" else 600)
    else:
        if path == "turn":
            c["tokens"] = _log(rng, 2, 500)
        c["context"] = _log(rng, 1, top)
        chunk = sizes[model].get("chunk", 0)
        if chunk:                                    # a turn that can be run again: it stays inside one chunk of positions
            c["context"] += max(0, chunk - c["context"] % chunk) if c["context"] % chunk + c["tokens"] > chunk else 0
    return c


# ---- inputs -------------------------------------------------------------------------------------------------------------

def _maker(seed):
    g = torch.Generator(device=DEV).manual_seed(seed * 7919 + 17)

    def rn(*shape, std=1.0, mean=0.0, dtype=torch.float16):
        return torch.empty(shape, dtype=dtype, device=DEV).normal_(mean, std, generator=g)
    return g, rn


def _rope(positions, dims, base=10000.0):
    """[n, dims / 2] angles in 64 bits."""
    f = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=DEV) / dims)
    return torch.as_tensor(positions, dtype=torch.float64, device=DEV).reshape(-1, 1) * f


def _neox_layer(rn, z):
    H, F = z["hidden"], z["ffn"]
    return dict(ln_w=rn(H, std=0.02, mean=1.0), ln_b=rn(H, std=0.01), w_qkv=rn(3 * H, H, std=0.02), b_qkv=rn(3 * H, std=0.01),
                w_o=rn(H, H, std=0.02), b_o=rn(H, std=0.01), post_ln_w=rn(H, std=0.02, mean=1.0), post_ln_b=rn(H, std=0.01),
                w_up=rn(F, H, std=0.02), b_up=rn(F, std=0.01), w_down=rn(H, F, std=0.02), b_down=rn(H, std=0.01))


def _neox_inputs(case, seed):
    z, S = NEOX[case["model"]], case["context"]
    _, rn = _maker(seed)
    H, rows, L = z["hidden"], S + 8, case.get("layers", 1)
    t = dict(layers=[_neox_layer(rn, z) for _ in range(L)], k=rn(L, rows, H), v=rn(L, rows, H))
    if case["path"] == "step":
        t.update(embed=rn(z["vocab"], H), head=rn(z["vocab"], H, std=0.02), fw=rn(H, std=0.02, mean=1.0), fb=rn(H, std=0.01), token=seed % z["vocab"])
    else:
        a = _rope([S], z["rotary_dim"])
        t.update(x=rn(1, H), cos=torch.cat([a, a], 1).cos().float().contiguous(), sin=torch.cat([a, a], 1).sin().float().contiguous())
    return t


def _llama_inputs(case, seed):
    z, S = LLAMA[case["model"]], case["context"]
    g, rn = _maker(seed)
    H, F, D = z["hidden"], z["ffn"], z["head_dim"]
    t = dict(qkv=rn(3 * H, H, std=0.02), o=rn(H, H, std=0.02), rms=rn(H, std=0.1, mean=1.0))
    if case["path"] == "batch":
        B = case["batch"]
        lens = torch.randint(max(1, S // 2), S + S // 2 + 1, (B,), generator=torch.Generator().manual_seed(seed)).tolist()
        total = sum(lens) + B
        pool = B * (S + S // 2 + 1) + 37
        a = _rope(list(range(2 * S + 2)), D)
        ends = torch.tensor([0] + [n + 1 for n in lens]).cumsum(0)
        t.update(lens=lens, x=rn(B, H), res=rn(B, H), k=rn(pool, H), v=rn(pool, H), cos_sin=torch.cat([a.cos(), a.sin()], 1).float().contiguous(),
                 indices=torch.randperm(pool, generator=g, device=DEV)[:total].int().contiguous(), indptr=ends.int().to(DEV),
                 positions=torch.tensor(lens, dtype=torch.int64, device=DEV))
        return t
    t.update(x=rn(1, H), k=rn(S, H), v=rn(S, H))
    a = _rope([S], D)
    a = torch.repeat_interleave(a, 2, 1) if case["path"] == "plain" else torch.cat([a, a], 1)
    t.update(cos=a.cos().float().contiguous(), sin=a.sin().float().contiguous())
    if case["path"] == "layer":
        t.update(rms2=rn(H, std=0.1, mean=1.0), gate_up=rn(2 * F, H, std=0.02), down=rn(H, F, std=0.02))
    return t


def _nibotar_config(case):
    z = NIBOTAR[case["model"]]
    mixer = dict(heads=z["heads"], kv_heads=z["kv_heads"], dim=z["dim"], vdim=z["vdim"], scale=z["dim"] ** -0.5, v_mix=True,
                 mask=dict(size=z["chunk"]), rot=dict(base=10000.0, dims=z["dim"]))
    layers = []
    for i in range(case["layers"]):
        if z.get("experts") and i:                   # (the first layer is a dense one of the active experts' size)
            mlp = dict(kind="moe", expert=dict(ff=z["ff"]), router=dict(experts=z["experts"], top=z["top"]), shared=dict(ff=z["shared"]))
        else:
            mlp = dict(kind="dense", ff=z["top"] * z["ff"] + z["shared"] if z.get("experts") else z["ff"])
        layers.append(dict(type="attention", mixer=mixer, mlp=mlp))
    return dict(architecture="Nibotar", width=z["width"], vocab=z["vocab"], norm=dict(eps=1e-6), postln_alpha=2.0, logit_softcap=15.0, layers=layers)


def _nibotar_weights(cfg, g, rn):
    W, V = cfg["width"], cfg["vocab"]
    w, out = {"embed": rn(V, W), "head": rn(V, W, std=0.02), "final.norm": rn(W, std=0.02)}, 0.02 * (2 * len(cfg["layers"])) ** -0.5
    for i, layer in enumerate(cfg["layers"]):
        m, f, p = layer["mixer"], layer["mlp"], f"l{i}."
        for n, rows in (("q", m["heads"] * m["dim"]), ("k", m["kv_heads"] * m["dim"]), ("v", m["kv_heads"] * m["vdim"])):
            w[p + f"mix.{n}"] = rn(rows, W, std=0.02)
            w[p + f"mix.{n}.b"] = rn(rows, std=0.02)
            if n != "v":
                w[p + f"mix.{n}.norm"] = rn(rows, std=0.05, mean=1.2)
        w[p + "mix.vmix"] = torch.tensor(0.5)
        w[p + "mix.sink"] = rn(m["heads"])
        w[p + "mix.o"] = rn(W, m["heads"] * m["vdim"], std=out)
        w[p + "norm1"], w[p + "norm2"] = rn(W, std=0.02), rn(W, std=0.02)
        if f["kind"] == "dense":
            w[p + "mlp.up"], w[p + "mlp.down"] = rn(f["ff"], W, std=0.02), rn(W, f["ff"], std=out)
            continue
        E, top, ff, sh = f["router"]["experts"], f["router"]["top"], f["expert"]["ff"], f["shared"]["ff"]
        gate, up, down = rn(E, ff, W, std=0.02), rn(E, ff, W, std=0.02), rn(E, W, ff, std=out)
        for e in range(E):
            w[p + f"mlp.e{e}.gate"], w[p + f"mlp.e{e}.up"], w[p + f"mlp.e{e}.down"] = gate[e], up[e], down[e]
        w[p + "mlp.shared.gate"], w[p + "mlp.shared.up"], w[p + "mlp.shared.down"] = rn(sh, W, std=0.02), rn(sh, W, std=0.02), rn(W, sh, std=out)
        w[p + "mlp.table"] = torch.rand(V, E, device=DEV, generator=g).argsort(1)[:, :top].int().contiguous()
    return w


def _kagapel_config(case):
    """Layers with a gate and scaled angles, layers with sinks, and layers that read the latents of the layer before them take
    turns."""
    z = KAGAPEL[case["model"]]
    layers = []
    for i in range(case["layers"]):
        kind = i % 4                                 # 0, 3: gated; 1: sinks; 2: sinks and the latents of the layer before it
        rot = dict(base=10000.0, dims=z["rot_dim"])
        if kind in (0, 3):
            rot["scaling"] = dict(factor=4.0, original=2048.0, fast=32.0, slow=1.0)
        m = dict(heads=z["heads"], dim=z["dim"], rot_dim=z["rot_dim"], vdim=z["vdim"], kv_rank=z["kv_rank"], scale=(z["dim"] + z["rot_dim"]) ** -0.5, rot=rot)
        if kind == 2:
            m["kv_from"] = i - 1
        layers.append(dict(type="latent_attention" if kind in (0, 3) else "latent_attention_2", mixer=m, mlp=dict(kind="dense", ff=z["ff"])))
    return dict(architecture="Kagapel", width=z["width"], vocab=z["vocab"], streams=z["streams"], norm=dict(eps=1e-6), logit_scale=1.5,
                max_positions=8192, layers=layers)


def _kagapel_weights(cfg, g, rn):
    W, V, n = cfg["width"], cfg["vocab"], cfg["streams"]
    w = {"embed": rn(V, W), "pos": rn(cfg["max_positions"], W, std=0.5), "head": rn(V, W, std=0.02), "final.norm": rn(W, std=0.02, mean=1.0)}
    out = 0.02 * (2 * len(cfg["layers"])) ** -0.5
    for i, layer in enumerate(cfg["layers"]):
        m, ff, p = layer["mixer"], layer["mlp"]["ff"], f"l{i}."
        H, D, R, Dv, r = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        w[p + "mix.q"] = rn(H * (D + R), W, std=0.02)
        if "kv_from" not in m:
            w[p + "mix.dkv"], w[p + "mix.dkv.norm"] = rn(r + R, W, std=0.02), rn(r, std=0.02, mean=1.0)
        w[p + "mix.uk"], w[p + "mix.uv"] = rn(H * D, r, std=0.04), rn(H * Dv, r, std=0.04)
        w[p + "mix.o"] = rn(W, H * Dv, std=out)
        if layer["type"] == "latent_attention":
            w[p + "mix.g"] = rn(H * Dv, W, std=0.02)
        else:
            w[p + "mix.sink"] = rn(H)
        w[p + "mlp.gate"], w[p + "mlp.up"], w[p + "mlp.down"] = rn(ff, W, std=0.02), rn(ff, W, std=0.02), rn(W, ff, std=out)
        w[p + "mlp.gate.b"], w[p + "mlp.up.b"], w[p + "mlp.down.b"] = rn(ff, std=0.02), rn(ff, std=0.02), rn(W, std=0.02)
        for q in (1, 2):
            w[p + f"norm{q}"] = rn(W, std=0.02, mean=1.0)
            w[p + f"hc{q}.in"], w[p + f"hc{q}.out"] = rn(n, std=0.02, mean=1.0 / n), rn(n, std=0.02, mean=1.0)
            w[p + f"hc{q}.mix"] = (torch.eye(n, device=DEV) * 0.9 + 0.02).to(w[p + "norm1"].dtype)
    return w


def _seq_inputs(case, seed):
    """Configuration, checkpoint tensors, and the tokens of the context and of the call."""
    g, raw = _maker(seed)
    dtype = torch.float32 if case["dtype"] == "f32" else torch.bfloat16

    def rn(*shape, std=1.0, mean=0.0):
        return raw(*shape, std=std, mean=mean, dtype=dtype)
    nib = case["family"] == "nibotar"
    cfg = _nibotar_config(case) if nib else _kagapel_config(case)
    w = (_nibotar_weights if nib else _kagapel_weights)(cfg, g, rn)
    tokens = torch.randint(0, cfg["vocab"], (case["context"] + case["tokens"],), generator=torch.Generator().manual_seed(seed + 1)).tolist()
    return cfg, w, tokens


def prepare(case, seed):
    if case["family"] == "neox":
        t = _neox_inputs(case, seed)
        if case["path"] == "step":
            import clusterfusionplus_amd as pkg
            z = NEOX[case["model"]]
            cfg = pkg.NeoxConfig(z["hidden"], z["heads"], z["head_dim"], z["rotary_dim"], z["ffn"], case["layers"], z["vocab"])
            t["decoder"] = pkg.NeoxDecoder(cfg, t["layers"], t["embed"], t["fw"], t["fb"], t["head"], list(t["k"]), list(t["v"]))
        else:
            import clusterfusion
            w = t["layers"][0]
            t["op"] = getattr(clusterfusion, case["model"] + ("_decoder_layer_split" if case["path"] == "layer_split" else "_decoder_layer"))
            t["args"] = [t["x"], w["w_qkv"], w["b_qkv"], w["w_o"], w["b_o"], t["k"][0], t["v"][0], w["ln_w"], w["ln_b"], t["cos"], t["sin"],
                         w["post_ln_w"], w["post_ln_b"], w["w_up"], w["b_up"], w["w_down"], w["b_down"], case["context"]]
        return dict(case=case, **t)
    if case["family"] == "llama":
        t = _llama_inputs(case, seed)
        if case["path"] == "batch":
            t.update(out=torch.empty_like(t["x"]), res_out=torch.empty_like(t["x"]),
                     kptr=torch.tensor([t["k"].data_ptr()], dtype=torch.uint64, device=DEV), vptr=torch.tensor([t["v"].data_ptr()], dtype=torch.uint64, device=DEV))
        return dict(case=case, **t)
    from clusterfusionplus_amd import kagapel, nibotar
    cfg, w, tokens = _seq_inputs(case, seed)
    n, S = case["tokens"], case["context"]
    make = nibotar.from_tensors if case["family"] == "nibotar" else kagapel.from_tensors
    dtype = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
    m = make(cfg, w, dtype, capacity=S + n + 16, max_portion=max(2048, n))
    del w
    if S:
        m.forward(0, tokens[:S], 0)
    return dict(case=case, model=m, tokens=tokens[S:], want=list(range(n)) if case["want"] == "all" else [n - 1])


def run(state):
    case = state["case"]
    if case["family"] == "neox":
        if case["path"] == "step":
            d = state["decoder"]
            d.set_state(state["token"], case["context"])
            d.graph_steps(1)
            return dict(logits=d.logits.clone(), hidden=d.hidden.clone(), k_caches=state["k"], v_caches=state["v"])
        out, k, v = state["op"](*state["args"])
        return dict(output=out, k=k, v=v, k_cache=state["k"], v_cache=state["v"])
    if case["family"] == "llama":
        import clusterfusion as cf
        s, z = state, LLAMA[case["model"]]
        if case["path"] == "batch":
            cf.llama_decoder_layer_batch_decode_sglang(s["out"], s["res_out"], s["x"], s["res"], s["qkv"], s["o"], s["indptr"], s["indices"],
                                                       s["kptr"], s["vptr"], 0, s["rms"], z["eps"], s["positions"], s["cos_sin"])
            return dict(output=s["out"], residual=s["res_out"], k_cache=s["k"], v_cache=s["v"])
        if case["path"] == "plain":
            out, k, v = cf.llama_decoder_layer(s["x"], s["qkv"], s["o"], s["k"], s["v"], s["rms"], s["cos"], s["sin"], z["heads"])
        else:
            out, k, v = cf.llama_decoder_layer_full(s["x"], s["qkv"], s["o"], s["k"], s["v"], s["rms"], s["rms2"], s["gate_up"], s["down"], z["eps"],
                                                    s["cos"], s["sin"], z["heads"])
        return dict(output=out, k=k, v=v)
    m = state["model"]
    if case["path"] == "step":
        m.set_state(state["tokens"][0], case["context"])
        m.graph_steps(1)
        return dict(logits=m.logits.clone())            # (the next step writes the model's own)
    return dict(logits=m.forward(0, state["tokens"], case["context"], state["want"]))


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------

def _expected_experts(experts, top, tokens):
    return experts * (1.0 - (1.0 - top / experts) ** tokens)


def work(case):
    S = case["context"]
    if case["family"] == "neox":
        z, L = NEOX[case["model"]], case.get("layers", 1)
        H, F = z["hidden"], z["ffn"]
        n = L * (4 * H * H + 2 * F * H)
        b = 2 * n + L * (2 * (9 * H + F) + 2 * S * H * 2 + 2 * H * 2)
        f = 2 * n + L * 4 * S * H
        if case["path"] == "step":
            n = z["vocab"] * H
            b, f = b + 2 * n + 4 * z["vocab"], f + 2 * n
        return dict(bytes=b, flops=f)
    if case["family"] == "llama":
        z, B = LLAMA[case["model"]], case.get("batch", 1)
        H, F = z["hidden"], z["ffn"]
        n = 4 * H * H + (3 * H * F if case["path"] == "layer" else 0)
        return dict(bytes=2 * n + B * (2 * S * H * 2 + 8 * H), flops=2 * B * n + B * 4 * S * H)
    z, T, L, e = SEQ[case["family"]][case["model"]], case["tokens"], case["layers"], 4 if case["dtype"] == "f32" else 2
    W, H, Dv, V = z["width"], z["heads"], z["vdim"], z["vocab"]
    wanted = T if case["want"] == "all" else 1
    read = used = 0                                  # matrix elements that are read, and that one token uses
    if case["family"] == "nibotar":
        G, D, c = z["kv_heads"], z["dim"], z["chunk"]
        row, per_pair = G * (D + Dv), 2 * H * (D + Dv)
        seen = sum(p % c + 1 for p in range(S, S + T))
        cached = min(S % c, S)
        for i in range(L):
            n = W * (H * D + G * D + G * Dv) + W * H * Dv
            if z.get("experts") and i:
                used += n + 3 * W * (z["top"] * z["ff"] + z["shared"])
                read += n + 3 * W * (_expected_experts(z["experts"], z["top"], T) * z["ff"] + z["shared"])
            else:
                n += 2 * W * (z["top"] * z["ff"] + z["shared"] if z.get("experts") else z["ff"])
                used, read = used + n, read + n
        cache_bytes = L * (cached + min(T, c)) * row * e
    else:
        D, R, r = z["dim"], z["rot_dim"], z["kv_rank"]
        seen, cached = sum(range(S + 1, S + T + 1)), S
        # keys and values of one head: made from the latents once per position, or the queries taken to the latents
        per_pair = 2 * H * (D + R + Dv)
        cache_bytes = 0
        for i in range(L):
            n = W * (H * (D + R) + (r + R if i % 4 != 2 else 0) + (H * Dv if i % 4 in (0, 3) else 0)) + H * (D + Dv) * r + W * H * Dv + 3 * W * z["ff"]
            used, read = used + n, read + n
            cache_bytes += (cached + (T if i % 4 != 2 else 0)) * (r + R) * e
    return dict(bytes=e * (read + V * W) + cache_bytes + 4 * wanted * V, flops=2 * T * used + 2 * wanted * V * W + L * per_pair * seen)


# ---- the same in 64 bits --------------------------------------------------------------------------------------------------

def _f(t):
    return t.double()


def _softmax_rows(s, extra=None):
    """Softmax over the last dimension; `extra`: one more term exp(extra) in the denominator."""
    top = s.amax(-1, keepdim=True)
    if extra is not None:
        top = torch.maximum(top, extra)
    p = s.sub_(top).exp_()
    den = p.sum(-1, keepdim=True)
    if extra is not None:
        den = den + (extra - top).exp()
    return p.div_(den)


def _layer_norm(x, w, b, eps=1e-5):
    m = x.mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(((x - m) ** 2).mean(-1, keepdim=True) + eps) * _f(w) + _f(b)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _halves(t, a, n):
    """The first n of the last dimension rotated, i with i + n / 2, by the angles a [n / 2]."""
    u, v, rest = t[..., :n // 2], t[..., n // 2:n], t[..., n:]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), rest], -1)


def _one_query(q, keys, vals):
    """q [heads, D], keys and values [S, heads, D]."""
    p = _softmax_rows((keys * q).sum(-1).T / math.sqrt(q.shape[1]))
    return (p.T[:, :, None] * vals).sum(0)


def _exact_neox(case, seed):
    z, t, S = NEOX[case["model"]], _neox_inputs(case, seed), case["context"]
    H, nh, D, R = z["hidden"], z["heads"], z["head_dim"], z["rotary_dim"]
    step = case["path"] == "step"
    x = _f(t["embed"][t["token"]])[None] if step else _f(t["x"])
    a = _rope([S], R)[0]
    kc, vc = _f(t["k"]), _f(t["v"])
    for i, w in enumerate(t["layers"]):
        n1, n2 = _layer_norm(x, w["ln_w"], w["ln_b"]), _layer_norm(x, w["post_ln_w"], w["post_ln_b"])
        q, k, v = (n1 @ _f(w["w_qkv"]).T + _f(w["b_qkv"])).reshape(nh, 3, D).unbind(1)
        q, k = _halves(q, a, R), _halves(k, a, R)
        kc[i, S], vc[i, S] = k.reshape(-1), v.reshape(-1)
        o = _one_query(q, kc[i, :S + 1].reshape(S + 1, nh, D), vc[i, :S + 1].reshape(S + 1, nh, D))
        u = n2 @ _f(w["w_up"]).T + _f(w["b_up"])
        u = 0.5 * u * (1 + torch.tanh(math.sqrt(2 / math.pi) * (u + 0.044715 * u ** 3)))
        x = x + o.reshape(1, H) @ _f(w["w_o"]).T + _f(w["b_o"]) + u @ _f(w["w_down"]).T + _f(w["b_down"])
    if step:
        return dict(logits=(_layer_norm(x, t["fw"], t["fb"]) @ _f(t["head"]).T).reshape(-1), hidden=x.reshape(-1), k_caches=kc, v_caches=vc)
    return dict(output=x, k=k[None], v=v[None], k_cache=kc, v_cache=vc)


def _exact_llama(case, seed):
    z, t = LLAMA[case["model"]], _llama_inputs(case, seed)
    H, nh, D = z["hidden"], z["heads"], z["head_dim"]

    def one(n, a, pairs, keys, vals):
        if pairs:
            wq, wk, wv = (w for w in t["qkv"].reshape(3, H, H))
            q, k, v = ((n @ _f(w)).reshape(nh, D) for w in (wq, wk, wv))
            rot = lambda y: torch.stack([y[:, 0::2] * a.cos() - y[:, 1::2] * a.sin(), y[:, 1::2] * a.cos() + y[:, 0::2] * a.sin()], -1).reshape(nh, D)  # noqa: E731
            q, k = rot(q), rot(k)
        else:
            q, k, v = (n @ _f(t["qkv"]).T).reshape(3, nh, D).unbind(0)
            q, k = _halves(q, a, D), _halves(k, a, D)
        o = _one_query(q, torch.cat([_f(keys).reshape(-1, nh, D), k[None]]), torch.cat([_f(vals).reshape(-1, nh, D), v[None]]))
        return (o.reshape(1, H) @ (_f(t["o"]) if pairs else _f(t["o"]).T)), k, v
    if case["path"] == "batch":
        r = _f(t["x"]) + _f(t["res"])
        n = _rms(_f(r.half()), z["eps"]) * _f(t["rms"])      # (the sum is a float16 tensor that the call returns)
        kc, vc, outs, at = _f(t["k"]), _f(t["v"]), [], 0
        for b, length in enumerate(t["lens"]):
            rows = t["indices"][at:at + length + 1].long()
            at += length + 1
            o, k, v = one(n[b:b + 1], _rope([length], D)[0], False, t["k"][rows[:-1]], t["v"][rows[:-1]])
            outs.append(o)
            kc[rows[-1]], vc[rows[-1]] = k.reshape(-1), v.reshape(-1)
        return dict(output=torch.cat(outs), residual=r, k_cache=kc, v_cache=vc)
    a = _rope([case["context"]], D)[0]
    x = _f(t["x"])
    o, k, v = one(_rms(x, 1e-6 if case["path"] == "plain" else z["eps"]) * _f(t["rms"]), a, case["path"] == "plain", t["k"], t["v"])
    if case["path"] == "layer":
        h = x + o
        g, u = ((_rms(h, z["eps"]) * _f(t["rms2"])) @ _f(t["gate_up"]).T).reshape(2, -1)
        o = h + (g * torch.sigmoid(g) * u)[None] @ _f(t["down"]).T
    return dict(output=o, k=k[None], v=v[None])


def _attend(q, k, v, scale, sink, first):
    """Causal attention of one head over positions that see back to `first` [T]; q, k [T, D], v [T, Dv]."""
    T, out = q.shape[0], torch.empty_like(v)
    j = torch.arange(T, device=DEV)
    for i0 in range(0, T, 2048):
        i = j[i0:i0 + 2048, None]
        hi = int(i[-1]) + 1
        lo = int(first[i0])
        s = (q[i0:hi] @ k[lo:hi].T) * scale
        s.masked_fill_((j[None, lo:hi] > i) | (j[None, lo:hi] < first[i0:hi, None]), -math.inf)
        out[i0:hi] = _softmax_rows(s, sink) @ v[lo:hi]
    return out


def _gated(h, gate, up, down, bg=0.0, bu=0.0, bd=0.0):
    g = h @ _f(gate).T + bg
    g = g * torch.sigmoid(g) * (h @ _f(up).T + bu)
    return g @ _f(down).T + bd


def _exact_nibotar(case, seed):
    cfg, w, tokens = _seq_inputs(case, seed)
    eps, T = cfg["norm"]["eps"], len(tokens)
    ids = torch.tensor(tokens, device=DEV)
    x, v_first, pos = _f(w["embed"][ids]), None, torch.arange(T, device=DEV)
    for i, layer in enumerate(cfg["layers"]):
        m, f, p = layer["mixer"], layer["mlp"], f"l{i}."
        H, G, D, Dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (x @ _f(w[p + f"mix.{n}"]).T + _f(w[p + f"mix.{n}.b"]) for n in "qkv")
        a = _rope(list(range(T)), m["rot"]["dims"])[:, None, :]

        def rotated(y, n, name):
            y = (_rms(y, eps) * _f(w[p + f"mix.{name}.norm"])).reshape(T, n, D)
            e, o = y[..., 0::2], y[..., 1::2]
            return torch.stack([e * a.cos() - o * a.sin(), o * a.cos() + e * a.sin()], -1).reshape(T, n, D)
        q, k = rotated(q, H, "q"), rotated(k, G, "k")
        if v_first is None:
            v_first = v
        else:
            lam = float(w[p + "mix.vmix"])
            v = (1 - lam) * v + lam * v_first
        first, vh = pos // m["mask"]["size"] * m["mask"]["size"], v.reshape(T, G, Dv)
        o = torch.empty(T, H, Dv, dtype=torch.float64, device=DEV)
        for h in range(H):
            g = h // (H // G)
            o[:, h] = _attend(q[:, h], k[:, g], vh[:, g].contiguous(), m["scale"], _f(w[p + "mix.sink"][h]), first)
        x = _rms(2.0 * x + o.reshape(T, -1) @ _f(w[p + "mix.o"]).T, eps) * (1 + _f(w[p + "norm1"]))
        if f["kind"] == "dense":
            y = torch.relu(x @ _f(w[p + "mlp.up"]).T).square_() @ _f(w[p + "mlp.down"]).T
        else:
            y, table, top = torch.zeros_like(x), w[p + "mlp.table"][ids], f["router"]["top"]
            for e in range(f["router"]["experts"]):
                at = (table == e).any(1).nonzero().reshape(-1)
                if at.numel():
                    y[at] += _gated(x[at], *(w[p + f"mlp.e{e}.{n}"] for n in ("gate", "up", "down"))) / top
            y += _gated(x, *(w[p + f"mlp.shared.{n}"] for n in ("gate", "up", "down")))
        x = _rms(2.0 * x + y, eps) * (1 + _f(w[p + "norm2"]))
    x = x[case["context"]:] if case["want"] == "all" else x[-1:]
    z = (_rms(x, eps) * (1 + _f(w["final.norm"]))) @ _f(w["head"]).T
    return 15.0 * torch.tanh(z / 15.0)


def _yarn(dims, base, sc):
    """Angle per position of every pair, and the factor on cos and sin."""
    f = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    if not sc:
        return torch.tensor(f, dtype=torch.float64, device=DEV), 1.0
    at = lambda turns: dims * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(base))  # noqa: E731
    lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), dims - 1)
    r = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
    f = [a / sc["factor"] * b + a * (1 - b) for a, b in zip(f, r)]
    return torch.tensor(f, dtype=torch.float64, device=DEV), 0.1 * math.log(sc["factor"]) + 1.0


def _exact_kagapel(case, seed):
    cfg, w, tokens = _seq_inputs(case, seed)
    eps, T, n = cfg["norm"]["eps"], len(tokens), cfg["streams"]
    pos = torch.arange(T, device=DEV)
    x = _f(w["embed"][torch.tensor(tokens, device=DEV)]) + _f(w["pos"][:T])
    xs, cached, none = [x.clone() for _ in range(n)], {}, torch.zeros_like(pos)

    def sublayer(p, q, f):
        nonlocal xs
        inn, mix, out = (_f(w[f"{p}hc{q}.{name}"]).tolist() for name in ("in", "mix", "out"))
        y = f(_rms(sum(a * b for a, b in zip(inn, xs)), eps) * _f(w[f"{p}norm{q}"]))
        xs = [sum(mix[a][b] * xs[a] for a in range(n)) + out[b] * y for b in range(n)]
    for i, layer in enumerate(cfg["layers"]):
        m, p = layer["mixer"], f"l{i}."
        H, D, R, Dv, r = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        freq, factor = _yarn(R, m["rot"]["base"], m["rot"].get("scaling"))
        a = pos[:, None] * freq

        def rotated(y):
            u, v = y[..., :R // 2], y[..., R // 2:]
            return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1) * factor

        def mixer(h):
            if "kv_from" in m:
                c, kr = cached[m["kv_from"]]
            else:
                z = h @ _f(w[p + "mix.dkv"]).T
                c, kr = cached[i] = _rms(z[:, :r], eps) * _f(w[p + "mix.dkv.norm"]), rotated(z[:, r:])
            q = (h @ _f(w[p + "mix.q"]).T).reshape(T, H, D + R)
            k, v = (c @ _f(w[p + "mix.uk"]).T).reshape(T, H, D), (c @ _f(w[p + "mix.uv"]).T).reshape(T, H, Dv)
            o = torch.empty(T, H, Dv, dtype=torch.float64, device=DEV)
            for j in range(H):
                sink = _f(w[p + "mix.sink"][j]) if p + "mix.sink" in w else None
                o[:, j] = _attend(torch.cat([q[:, j, :D], rotated(q[:, j, D:])], 1), torch.cat([k[:, j], kr], 1), v[:, j].contiguous(), m["scale"], sink, none)
            o = o.reshape(T, -1)
            if p + "mix.g" in w:
                o = o * torch.sigmoid(h @ _f(w[p + "mix.g"]).T)
            return o @ _f(w[p + "mix.o"]).T
        sublayer(p, 1, mixer)
        sublayer(p, 2, lambda h: _gated(h, *(w[f"{p}mlp.{s}"] for s in ("gate", "up", "down")), *(_f(w[f"{p}mlp.{s}.b"]) for s in ("gate", "up", "down"))))
    x = sum(xs)
    x = x[case["context"]:] if case["want"] == "all" else x[-1:]
    return (_rms(x, eps) * _f(w["final.norm"])) @ _f(w["head"]).T * cfg["logit_scale"]


def exact(case, seed):
    with torch.no_grad():
        if case["family"] == "neox":
            return _exact_neox(case, seed)
        if case["family"] == "llama":
            return _exact_llama(case, seed)
        z = (_exact_nibotar if case["family"] == "nibotar" else _exact_kagapel)(case, seed)
        return dict(logits=z.reshape(-1) if case["path"] == "step" else z)


def tolerance(case):
    """About four times the error against 64 bits that the data types cause."""
    if case["family"] in ("neox", "llama"):
        return {"rel": 4e-3}
    return {"rel": 1e-5} if case["dtype"] == "f32" else {"rel": 0.03}
