"""Workloads whose speed is measured: steps of models served through ``Engine.step``.

A case is one batch that a server runs: decoded tokens of requests whose context lies in the cache, prompts
(or portions of them behind cached tokens), or both in one step (``mode`` "step"); or whole requests, prompt and
then a few decoded tokens, from admission to release (``mode`` "request").  Models are four layers (two with 128
experts) of the sizes that ``bench.py`` measures, with a vocabulary of 32,768, so that the layers and not the
output table carry the time as they do in a whole model; weights, prompts and contexts are drawn from a seed.

``exact`` computes the same logits with plain torch in 64 bits: whole sequences, no cache, no shared code.
"""
from __future__ import annotations

import math
import zlib

import torch

from spite_amd import Engine, StepEntry

DEVICE = "cuda:0"
VOCAB = 32768
PORTION = 2048            # the scheduler's token budget of a step
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}

# width, heads, experts, and (Llama 4) expert width, dense width, a layer with experts every n, layers
LLAMA4 = {
    "scout": dict(width=5120, heads=40, kv_heads=8, experts=16, expert_ff=8192, dense_ff=16384, moe_every=1, layers=4),
    # the same layers, 128 experts in every second one
    "many": dict(width=5120, heads=40, kv_heads=8, experts=128, expert_ff=8192, dense_ff=16384, moe_every=2, layers=2),
    # a small model of the same kind
    "2k": dict(width=2048, heads=16, kv_heads=4, experts=16, expert_ff=3072, dense_ff=6144, moe_every=1, layers=4),
}
# the other designs: width, heads, experts, experts a token, expert and shared widths
DESIGNS = {
    "2k": dict(width=2048, heads=16, experts=16, top=4, expert_ff=1024, shared_ff=2048, layers=4),
    "5k": dict(width=5120, heads=40, experts=16, top=2, expert_ff=4096, shared_ff=8192, layers=4),
}


# ------------------------------------------------------------------ the cases
def _case(name, model="llama4", size="scout", dtype="bfloat16", mode="step", decoding=0, context=0, apart=0, prompts=0,
          prompt=0, prompt_apart=0, past=0, want="last", then=0):
    """``decoding`` requests with ``context``, ``context - apart``, ... cached tokens bring one token each;
    ``prompts`` requests bring ``prompt``, ``prompt - prompt_apart``, ... tokens behind ``past`` cached ones and want
    the logits of the last place or of all; in mode "request" every one decodes ``then`` further tokens."""
    c = dict(model=model, size=size, dtype=dtype, mode=mode, decoding=decoding, context=context, apart=apart,
             prompts=prompts, prompt=prompt, prompt_apart=prompt_apart, past=past, want=want, then=then)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # one user of a small model, a token at a time: launches and latency
        _case("small-decode-1", size="2k", decoding=1, context=517),
        # the headline's model: one user, the headline batch, a full server with contexts of every length
        _case("decode-1", decoding=1, context=4096),
        _case("decode-8", decoding=8, context=4096),
        _case("decode-64-ragged", decoding=64, context=1537, apart=17),
        # few requests with long contexts (past the chunk of 8,192 on the rotating layers)
        _case("decode-long", decoding=4, context=14003, apart=1201),
        # prompts: the headline's 2,048 tokens; a few short ones that arrive together
        _case("prefill-2048", prompts=1, prompt=2048),
        _case("prefill-short", prompts=3, prompt=157, prompt_apart=47),
        # a server's mixed step: decoded tokens lead a portion of a prompt behind cached tokens
        _case("mixed", decoding=16, context=1211, apart=31, prompts=1, prompt=1531, past=2048),
        # 128 experts, a batch of decoding requests: nearly every token meets an expert of its own
        _case("many-experts-decode-32", size="many", decoding=32, context=1019, apart=13),
        # the 32-bit path: the logits of every place of a short text, then a few tokens, as a replay asks for them
        _case("fp32-replay", size="2k", dtype="float32", mode="request", prompts=1, prompt=301, want="all", then=4),
        # attention over a cached latent: two prompts and their first tokens
        _case("latent-request", model="ravenex", size="5k", mode="request", prompts=2, prompt=1021, prompt_apart=256, then=4),
        # linear attention with a state per request beside attention with sinks: a prompt and its first tokens
        _case("linear-request", model="tebalorn", size="2k", mode="request", prompts=1, prompt=1531, then=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "small", "many", "prefill", "prefill", "mixed", "fp32", "latent", "linear"])
    if kind in ("decode", "small", "many"):
        size = {"decode": "scout", "small": "2k", "many": "many"}[kind]
        n = _log(rng, 1, 64 if kind == "decode" else 32)
        context = _log(rng, 64, min(16000, 56000 // n if kind == "decode" else 32000 // n))
        return _case(None, size=size, decoding=n, context=context, apart=rng.randint(0, context // (2 * n)))
    if kind == "prefill":
        m = rng.randint(1, 4)
        p = _log(rng, 16, 2048 // m)
        return _case(None, size=rng.choice(["scout", "scout", "2k"]), prompts=m, prompt=p, prompt_apart=rng.randint(0, p // (2 * m)),
                     past=rng.choice([0, 0, _log(rng, 64, 4096)]))
    if kind == "mixed":
        n, context = _log(rng, 1, 32), _log(rng, 64, 1600)
        return _case(None, decoding=n, context=context, apart=rng.randint(0, context // (2 * n)), prompts=1,
                     prompt=_log(rng, 32, 2000), past=rng.choice([0, _log(rng, 64, 4096)]))
    if kind == "fp32":
        return _case(None, size="2k", dtype="float32", mode="request", prompts=1, prompt=_log(rng, 16, 320),
                     want=rng.choice(["last", "all"]), then=rng.randint(1, 6))
    m = rng.randint(1, 3)
    p = _log(rng, 64, 2048 // m)
    return _case(None, model="ravenex" if kind == "latent" else "tebalorn", size=rng.choice(["2k", "5k"]), mode="request",
                 prompts=m, prompt=p, prompt_apart=rng.randint(0, p // (2 * m)), then=rng.randint(1, 6))


# ------------------------------------------------------------------ models
def _config(c):
    if c["model"] == "llama4":
        s = LLAMA4[c["size"]]
        return dict(
            architectures=["Llama4ForCausalLM"], num_hidden_layers=s["layers"], hidden_size=s["width"],
            num_attention_heads=s["heads"], num_key_value_heads=s["kv_heads"], head_dim=128, rms_norm_eps=1e-5,
            num_local_experts=s["experts"], num_experts_per_tok=1, intermediate_size=s["expert_ff"],
            intermediate_size_mlp=s["dense_ff"], interleave_moe_layer_step=s["moe_every"], vocab_size=VOCAB,
            tie_word_embeddings=False, rope_theta=500000.0,
            rope_scaling=dict(rope_type="llama3", factor=16.0, low_freq_factor=1.0, high_freq_factor=4.0,
                              original_max_position_embeddings=8192),
            attention_chunk_size=8192, use_qk_norm=True, attn_temperature_tuning=True, floor_scale=8192, attn_scale=0.1,
            torch_dtype=c["dtype"])
    s = DESIGNS[c["size"]]
    H = s["heads"]
    mlp = {"kind": "moe", "router": {"experts": s["experts"], "top": s["top"]}, "expert": {"ff": s["expert_ff"]},
           "shared": {"ff": s["shared_ff"]}}
    both = {"vocab": VOCAB, "width": s["width"], "norm": {"eps": 1e-6}, "token_side": {"dim": 256}, "torch_dtype": c["dtype"]}
    if c["model"] == "ravenex":       # a layer with a cache and one that reads it, in turn
        mixer = {"heads": H, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "mask": {"size": 4096},
                 "rot": {"base": 10000.0, "dims": 64}, "scale": 192 ** -0.5}
        return dict(both, architecture="Ravenex", residual_mult=0.7,
                    layers=[{"type": "latent_attention", "mixer": dict(mixer, **({"kv_from": i - 1} if i % 2 else {})), "mlp": mlp}
                            for i in range(s["layers"])])
    linear = {"heads": H, "dim": 128, "vdim": 128}
    decays = lambda a, b: [1.0 - 2.0 ** (-a - b * h / (H - 1)) for h in range(H)]
    mixers = [("gla", dict(linear, tau=8.0)), ("lightning", dict(linear, decay=decays(5.0, 3.0))),
              ("attention", {"heads": H, "kv_heads": H // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": 4096},
                             "rot": {"base": 1000000.0, "dims": 64,
                                     "scaling": {"factor": 4.0, "original": 8192, "fast": 16.0, "slow": 2.0}}}),
              ("lightning", dict(linear, decay=decays(4.0, 4.0)))]
    return dict(both, architecture="Tebalorn", embedding={"scale": 8.0}, logit_scale=0.5,
                layers=[{"type": mixers[i][0], "mixer": mixers[i][1], "mlp": mlp} for i in range(s["layers"])])


def _llama4_shapes(cfg):
    d, L, E, F = cfg["hidden_size"], cfg["num_hidden_layers"], cfg["num_local_experts"], cfg["intermediate_size"]
    q, kv = cfg["num_attention_heads"] * 128, cfg["num_key_value_heads"] * 128
    out = {"model.embed_tokens.weight": (VOCAB, d), "lm_head.weight": (VOCAB, d), "model.norm.weight": (d,)}
    for i in range(L):
        p = f"model.layers.{i}."
        out[p + "input_layernorm.weight"] = out[p + "post_attention_layernorm.weight"] = (d,)
        for k, n in (("q", q), ("k", kv), ("v", kv)):
            out[p + f"self_attn.{k}_proj.weight"] = (n, d)
        out[p + "self_attn.o_proj.weight"] = (d, q)
        f, step = p + "feed_forward.", cfg["interleave_moe_layer_step"]
        inner = cfg["intermediate_size_mlp"]
        if (i + 1) % step == 0:
            out[f + "router.weight"] = (E, d)
            out[f + "experts.gate_up_proj"], out[f + "experts.down_proj"] = (E, d, 2 * F), (E, F, d)
            f, inner = f + "shared_expert.", F
        out[f + "gate_proj.weight"] = out[f + "up_proj.weight"] = (inner, d)
        out[f + "down_proj.weight"] = (d, inner)
    return out


def _design_shapes(cfg):
    d, side, L = cfg["width"], cfg["token_side"]["dim"], len(cfg["layers"])
    out = {"embed": (VOCAB, d), "side.embed": (VOCAB, L * side), "final.norm": (d,), "head": (VOCAB, d)}
    for i, layer in enumerate(cfg["layers"]):
        p, mx, ml = f"l{i}.", layer["mixer"], layer["mlp"]
        H, n, v = mx["heads"], mx["dim"], mx["vdim"]
        for k in ("norm1", "norm1b", "norm2", "norm2b") if layer["type"] == "latent_attention" else ("norm1",):
            out[p + k] = (d,)
        m = p + "mix."
        out[m + "o"] = (d, H * v)
        if layer["type"] == "latent_attention":
            r, R = mx["rot_dim"], mx["kv_rank"]
            out[m + "q"], out[m + "uk"], out[m + "uv"] = (H * (n + r), d), (H * n, R), (H * v, R)
            if "kv_from" not in mx:
                out[m + "dkv"], out[m + "dkv.norm"] = (R + r, d), (R,)
        else:
            G = mx.get("kv_heads", H)
            out[m + "q"], out[m + "k"], out[m + "v"] = (H * n, d), (G * n, d), (G * v, d)
            if layer["type"] == "attention":
                out[m + "sink"] = (H,)
            else:
                out[m + "g"], out[m + "norm"] = (H * v, d), ((v,) if layer["type"] == "gla" else (H * v,))
            if layer["type"] == "gla":
                out[m + "a1"], out[m + "a2"], out[m + "a2.b"] = (16, d), (H * n, 16), (H * n,)
        f, E = p + "mlp.", ml["router"]["experts"]
        out[f + "router"] = (E, d)
        if layer["type"] == "latent_attention":
            out[f + "correction"] = (E,)
        for k, ff in [(f"e{e}.", ml["expert"]["ff"]) for e in range(E)] + [("shared.", ml["shared"]["ff"])]:
            out[f + k + "gate"] = out[f + k + "up"] = (ff, d)
            out[f + k + "down"] = (d, ff)
        out[p + "side.gate"], out[p + "side.proj"], out[p + "side.norm"] = (side, d), (d, side), (d,)
    return out


_SMALL = ("correction", "sink", "a2.b")


def _generator(seed, name):
    return torch.Generator(device=DEVICE).manual_seed((int(seed) << 32) ^ zlib.crc32(name.encode()))


def _weights(cfg, dtype, seed):
    """The checkpoint: matrices N(0, 0.02), what leaves a sublayer smaller by the root of twice the layers, norm
    weights about 1, embedding rows that carry the stream.  Routers know their tokens, as trained ones do: a token's
    embedding leans towards the rows of the experts that are its own in each layer (drawn evenly), so that the choice
    is seldom a matter of rounding."""
    llama = "hidden_size" in cfg
    shapes = _llama4_shapes(cfg) if llama else _design_shapes(cfg)
    L, d = (cfg["num_hidden_layers"], cfg["hidden_size"]) if llama else (len(cfg["layers"]), cfg["width"])
    rows = 2.0 / (1.0 if llama else cfg.get("embedding", {"scale": 1.0})["scale"])
    top = 1 if llama else cfg["layers"][0]["mlp"]["router"]["top"]
    out, embed = {}, None
    for name, shape in shapes.items():
        base = name[:-7] if name.endswith(".weight") else name
        mean, std = 0.0, 0.02
        if base in ("model.embed_tokens", "embed"):
            embed, std = name, rows
        elif base == "side.embed":
            std = 1.0
        elif len(shape) == 1 and not base.endswith(_SMALL):
            mean = 1.0
        elif base.endswith("router"):
            std = 0.7 / math.sqrt(d)
        elif base.endswith((".o_proj", "down_proj", ".o", ".down")):
            std = 0.02 / math.sqrt(2 * L)
        out[name] = torch.empty(shape, dtype=dtype, device=DEVICE).normal_(mean, std, generator=_generator(seed, name))
    lean = torch.zeros((VOCAB, d), dtype=torch.float32, device=DEVICE)
    for name, r in out.items():
        if "router" in name:
            E = r.shape[0]
            r = r.float() / r.float().norm(dim=1, keepdim=True)
            own = torch.rand((VOCAB, E), device=DEVICE, generator=_generator(seed, name + " tokens")).topk(top, dim=1).indices
            for j in range(top):
                lean += r[own[:, j]]
    out[embed] = (out[embed].float() + 6.0 * rows * lean).to(dtype)
    return out


# ------------------------------------------------------------------ batches
def _requests(c):
    """(cached tokens, tokens of this step, places whose logits are wanted) of every request."""
    out = [(max(1, c["context"] - i * c["apart"]), 1, 1) for i in range(c["decoding"])]
    for i in range(c["prompts"]):
        n = max(1, c["prompt"] - i * c["prompt_apart"])
        out.append((c["past"], n, n if c["want"] == "all" else 1))
    return out


def _tokens(c, seed):
    """The whole token sequence of every request, whatever decodes afterwards included."""
    g = torch.Generator().manual_seed(int(seed) ^ 0x5EED)
    return [torch.randint(0, VOCAB, (past + n + c["then"],), generator=g).tolist() for past, n, _ in _requests(c)]


def prepare(case, seed):
    cfg, reqs, toks = _config(case), _requests(case), _tokens(case, seed)
    total = sum((len(t) + 63) // 64 * 64 + 64 for t in toks)
    eng = Engine(cfg, dtype=case["dtype"], tensors=_weights(cfg, DTYPES[case["dtype"]], seed), cache_tokens=total,
                 max_batch_tokens=PORTION, max_requests=len(reqs), device=DEVICE)
    if case["mode"] == "request":
        return {"case": case, "engine": eng, "requests": reqs, "tokens": toks}
    # the contexts, fed as the scheduler feeds them: portions of several requests in one step
    slots, batch, room = [eng.admit() for _ in reqs], [], PORTION
    for (past, _, _), t, slot in zip(reqs, toks, slots):
        at = 0
        while at < past:
            n = min(room, past - at)
            batch.append(StepEntry(slot, t[at:at + n]))
            at, room = at + n, room - n
            if room == 0:
                eng.step(batch)
                batch, room = [], PORTION
    if batch:
        eng.step(batch)
    entries = [StepEntry(s, t[past:past + n], list(range(n - w, n))) for (past, n, w), t, s in zip(reqs, toks, slots)]
    for _ in range(2):        # a running server has met steps of this shape before
        eng.step(entries, commit=False)
    return {"case": case, "engine": eng, "entries": entries}


def run(state):
    """One step of the batch (its positions stay uncommitted, so the next pass is the same step again), or whole
    requests from admission to release; the logits of every wanted place."""
    eng = state["engine"]
    if "entries" in state:
        return eng.step(state["entries"], commit=False)
    reqs, toks = state["requests"], state["tokens"]
    slots, out = [eng.admit() for _ in reqs], []
    out.append(eng.step([StepEntry(s, t[:n], list(range(n - w, n))) for (_, n, w), t, s in zip(reqs, toks, slots)]).clone())
    for k in range(state["case"]["then"]):
        out.append(eng.step([StepEntry(s, [t[n + k]], [0]) for (_, n, _), t, s in zip(reqs, toks, slots)]).clone())
    for s in slots:
        eng.release(s)
    return out


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """Bytes: every weight that the tokens use once (an expert if, on average, some token takes it), the keys and
    values that they see and write once a step, the logits.  FLOPs: the products of every token, scores and values."""
    cfg, reqs, item = _config(case), _requests(case), 4 if case["dtype"] == "float32" else 2
    steps = [[(past, n, w) for past, n, w in reqs]] + [[(past + n + k, 1, 1) for past, n, _ in reqs] for k in range(case["then"])]
    nbytes = flops = 0.0
    for step in steps:
        b, f = _step_work(cfg, case, step, item)
        nbytes, flops = nbytes + b, flops + f
    return {"bytes": nbytes, "flops": flops}


def _pairs(past, n, span, kind):
    """(keys seen by ``n`` queries behind ``past`` tokens, distinct keys read)."""
    if span is None:
        return n * past + n * (n + 1) / 2, past + n
    seen, first = 0, past
    for p in range(past, past + n):
        lo = p // span * span if kind == "chunk" else max(0, p - span + 1)
        seen, first = seen + p - lo + 1, min(first, lo)
    return seen, past + n - first


def _step_work(cfg, case, step, item):
    T, rows = sum(n for _, n, _ in step), sum(w for _, _, w in step)
    shapes = _llama4_shapes(cfg) if "hidden_size" in cfg else _design_shapes(cfg)
    llama = "hidden_size" in cfg
    E = cfg["num_local_experts"] if llama else cfg["layers"][0]["mlp"]["router"]["experts"]
    top = 1 if llama else cfg["layers"][0]["mlp"]["router"]["top"]
    touched = 1.0 - (1.0 - top / E) ** T
    b = f = 0.0
    for name, shape in shapes.items():
        n = math.prod(shape)
        if name in ("model.embed_tokens.weight", "embed", "side.embed"):
            b += T * shape[1] * item
        elif name in ("lm_head.weight", "head"):
            b, f = b + n * item, f + 2.0 * n * rows
        elif ".experts." in name:
            b, f = b + n * item * touched, f + 2.0 * n / E * T
        elif ".mlp.e" in name:
            b, f = b + n * item * touched, f + 2.0 * n * T * top / E
        else:
            b, f = b + n * item, f + (2.0 * n * T if len(shape) == 2 else 0.0)
    for past, n, _ in step:
        if llama:
            for i in range(cfg["num_hidden_layers"]):
                seen, keys = _pairs(past, n, cfg["attention_chunk_size"] if (i + 1) % 4 else None, "chunk")
                b += (keys + n) * 2 * cfg["num_key_value_heads"] * 128 * item
                f += 4.0 * seen * cfg["num_attention_heads"] * 128
            continue
        for layer in cfg["layers"]:
            mx = layer["mixer"]
            if layer["type"] in ("gla", "lightning"):         # the state once in and once out; k v^T and S q
                state = mx["heads"] * mx["dim"] * mx["vdim"]
                b, f = b + 8.0 * state, f + 5.0 * state * n
                continue
            seen, keys = _pairs(past, n, mx["mask"]["size"], "chunk" if layer["type"] == "attention" else "window")
            if layer["type"] == "attention":
                b += (keys + n) * mx["kv_heads"] * (mx["dim"] + mx["vdim"]) * item
                f += 2.0 * seen * mx["heads"] * (mx["dim"] + mx["vdim"])
            else:                                             # keys and values formed per head from the latent, as in the formulas
                b += (keys + ("kv_from" not in mx) * n) * (mx["kv_rank"] + mx["rot_dim"]) * item
                f += 2.0 * seen * mx["heads"] * (mx["dim"] + mx["rot_dim"] + mx["vdim"])
    return b + rows * VOCAB * 4, f


def tolerance(case):
    """Four times what the logits are off the 64-bit ones.  bfloat16: activations of 8 bits through four layers, 0.003
    to 0.006.  32-bit: sums of a few thousand terms in some order, 1e-6 to 2e-6."""
    return {"rel": 1e-5} if case["dtype"] == "float32" else {"rel": 0.02}


# ------------------------------------------------------------------ the same in 64 bits
F64 = torch.float64


def _mm(x, w):
    return x @ w.to(F64).T


def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _turn(x, pos, freq, adjacent=False, mag=1.0):
    """Pairs of the first 2 * len(freq) elements of every head turn by position * frequency."""
    half = freq.numel()
    ang = (pos.to(F64)[:, None] * freq).unsqueeze(1)
    c, s = torch.cos(ang) * mag, torch.sin(ang) * mag
    y = x.clone()
    ia, ib = (slice(0, 2 * half, 2), slice(1, 2 * half, 2)) if adjacent else (slice(0, half), slice(half, 2 * half))
    a, b = x[..., ia], x[..., ib]
    y[..., ia], y[..., ib] = a * c - b * s, b * c + a * s
    return y


def _attend(q, k, v, scale, kind=None, span=None, sink=None, block=512):
    """Causal attention of one whole sequence: q [T, H, D], k [T, G, D], v [T, G, V]."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    pos = torch.arange(T, device=q.device)
    out = torch.empty((T, H, v.shape[-1]), dtype=F64, device=q.device)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous()
    for a in range(0, T, block):
        b = min(a + block, T)
        lo = 0 if kind is None else a // span * span if kind == "chunk" else max(0, a - span + 1)
        i, j = pos[a:b, None], pos[None, lo:b]
        ok = j <= i
        if kind == "chunk":
            ok = ok & (j // span == i // span)
        elif kind == "window":
            ok = ok & (i - j < span)
        qb = q[a:b].transpose(0, 1).reshape(G, H // G * (b - a), -1)
        s = (torch.bmm(qb, kt[:, :, lo:b].contiguous()) * scale).view(H, b - a, b - lo).masked_fill(~ok, float("-inf"))
        m = s.amax(-1, keepdim=True)
        if sink is not None:
            m = torch.maximum(m, sink.view(H, 1, 1))
        p = torch.exp(s - m)
        z = p.sum(-1, keepdim=True)
        if sink is not None:
            z = z + torch.exp(sink.view(H, 1, 1) - m)
        o = torch.bmm((p / z).view(G, H // G * (b - a), b - lo), vt[:, lo:b].contiguous())
        out[a:b] = o.view(H, b - a, -1).transpose(0, 1)
    return out


def _each(seqs, fn):
    """``fn`` over the rows of every sequence, joined again."""
    return torch.cat([fn(a, b) for a, b in seqs])


def _llama4_freq(cfg):
    f = cfg["rope_theta"] ** (-torch.arange(64, dtype=F64, device=DEVICE) / 64)
    sc = cfg["rope_scaling"]
    orig, wave = sc["original_max_position_embeddings"], 2.0 * math.pi / f
    s = ((orig / wave - sc["low_freq_factor"]) / (sc["high_freq_factor"] - sc["low_freq_factor"])).clamp(0.0, 1.0)
    return (1.0 - s) * f / sc["factor"] + s * f


def _llama4_exact(cfg, W, tok, pos, seqs, rows):
    H, G, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["rms_norm_eps"]
    x, freq = W["model.embed_tokens.weight"][tok].to(F64), _llama4_freq(cfg)
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        n = _unit(x, eps) * W[p + "input_layernorm.weight"].to(F64)
        q, k, v = (_mm(n, W[p + f"self_attn.{z}_proj.weight"]).view(len(tok), -1, 128) for z in "qkv")
        kind = None
        if (i + 1) % 4:
            q, k, kind = _unit(_turn(q, pos, freq), eps), _unit(_turn(k, pos, freq), eps), "chunk"
        else:
            t = torch.log((pos + 1).div(cfg["floor_scale"], rounding_mode="floor").to(F64) + 1.0) * cfg["attn_scale"] + 1.0
            q = q * t[:, None, None]
        o = _each(seqs, lambda a, b: _attend(q[a:b], k[a:b], v[a:b], 128 ** -0.5, kind, cfg["attention_chunk_size"]))
        x = x + _mm(o.reshape(len(tok), H * 128), W[p + "self_attn.o_proj.weight"])
        del n, q, k, v, o
        n = _unit(x, eps) * W[p + "post_attention_layernorm.weight"].to(F64)
        f = p + "feed_forward."
        if f + "router.weight" in W:
            z = _mm(n, W[f + "router.weight"])
            best = z.argmax(-1)
            inner = cfg["intermediate_size"]
            for e in best.unique().tolist():
                sel = (best == e).nonzero()[:, 0]
                gu = (n[sel] * torch.sigmoid(z[sel, e])[:, None]) @ W[f + "experts.gate_up_proj"][e].to(F64)
                x[sel] += (_silu(gu[:, :inner]) * gu[:, inner:]) @ W[f + "experts.down_proj"][e].to(F64)
            f += "shared_expert."
        a = _silu(_mm(n, W[f + "gate_proj.weight"])) * _mm(n, W[f + "up_proj.weight"])
        x = x + _mm(a, W[f + "down_proj.weight"])
    return _mm(_unit(x[rows], eps) * W["model.norm.weight"].to(F64), W["lm_head.weight"])


def _experts_exact(n, W, f, ml, softmax):
    top = ml["router"]["top"]
    z = _mm(n, W[f + "router"])
    if softmax:
        val, idx = torch.topk(z, top, dim=-1)
        w = torch.softmax(val, dim=-1)
    else:
        s = torch.sigmoid(z)
        idx = torch.topk(s + W[f + "correction"].to(F64), top, dim=-1).indices
        w = s.gather(1, idx)
    glu = lambda x, p: _mm(_silu(_mm(x, W[p + "gate"])) * _mm(x, W[p + "up"]), W[p + "down"])
    out = glu(n, f + "shared.")
    for e in range(ml["router"]["experts"]):
        at, which = (idx == e).nonzero(as_tuple=True)
        if at.numel():
            out[at] += glu(n[at], f"{f}e{e}.") * w[at, which][:, None]
    return out


def _ravenex_exact(cfg, W, tok, pos, seqs, rows):
    eps, m, side = cfg["norm"]["eps"], cfg["residual_mult"], cfg["token_side"]["dim"]
    x, T = W["embed"][tok].to(F64), len(tok)
    for i, layer in enumerate(cfg["layers"]):
        p, mx = f"l{i}.", layer["mixer"]
        w = lambda name: W[p + name].to(F64)
        H, n_, r, R = mx["heads"], mx["dim"], mx["rot_dim"], mx["kv_rank"]
        freq = mx["rot"]["base"] ** (-2.0 * torch.arange(r // 2, dtype=F64, device=DEVICE) / r)
        n = _unit(x, eps) * w("norm1")
        if "kv_from" not in mx:
            z = _mm(n, w("mix.dkv"))
            latent, turned = _unit(z[:, :R], eps) * w("mix.dkv.norm"), _turn(z[:, None, R:], pos, freq, True)
        q = _mm(n, w("mix.q")).view(T, H, n_ + r)
        q = torch.cat([q[..., :n_], _turn(q[..., n_:], pos, freq, True)], -1)
        k = torch.cat([_mm(latent, w("mix.uk")).view(T, H, n_), turned.expand(T, H, r)], -1)
        v = _mm(latent, w("mix.uv")).view(T, H, -1)
        o = _each(seqs, lambda a, b: _attend(q[a:b], k[a:b], v[a:b], mx["scale"], "window", mx["mask"]["size"]))
        x = x + m * _unit(_mm(o.reshape(T, -1), w("mix.o")), eps) * w("norm1b")
        f = _experts_exact(_unit(x, eps) * w("norm2"), W, p + "mlp.", layer["mlp"], False)
        x = x + m * _unit(f, eps) * w("norm2b")
        e = W["side.embed"][tok, i * side:(i + 1) * side].to(F64)
        x = x + m * _unit(_mm(_gelu(_mm(x, w("side.gate"))) * e, w("side.proj")), eps) * w("side.norm")
    return _mm(_unit(x[rows], eps) * W["final.norm"].to(F64), W["head"])


def _recurrence(q, k, v, decay):
    """o_t = S_t^T q_t with S_t = diag(decay_t) S_(t-1) + k_t v_t^T, token by token."""
    T, H, D = q.shape
    S = torch.zeros((H, D, v.shape[-1]), dtype=F64, device=q.device)
    out = torch.empty_like(v)
    for t in range(T):
        S = torch.baddbmm(S.mul_(decay[t].unsqueeze(-1)), k[t].unsqueeze(-1), v[t].unsqueeze(1))
        out[t] = torch.bmm(q[t].unsqueeze(1), S)[:, 0]
    return out


def _yarn(rot):
    dims, base, sc = rot["dims"], rot["base"], rot["scaling"]
    i = torch.arange(dims // 2, dtype=F64, device=DEVICE)
    f = base ** (-2.0 * i / dims)
    index = lambda turns: dims * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(index(sc["fast"])), 0), min(math.ceil(index(sc["slow"])), dims - 1)
    r = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return (1.0 - r) * f + r * f / sc["factor"], 0.1 * math.log(sc["factor"]) + 1.0


def _tebalorn_exact(cfg, W, tok, pos, seqs, rows):
    eps, side, T = cfg["norm"]["eps"], cfg["token_side"]["dim"], len(tok)
    x = W["embed"][tok].to(F64) * cfg["embedding"]["scale"]
    for i, layer in enumerate(cfg["layers"]):
        p, mx, kind = f"l{i}.", layer["mixer"], layer["type"]
        w = lambda name: W[p + name].to(F64)
        H, D = mx["heads"], mx["dim"]
        n = _unit(x, eps) * w("norm1")
        q, k, v = (_mm(n, w("mix." + z)).view(T, -1, D) for z in "qkv")
        if kind == "attention":
            freq, mag = _yarn(mx["rot"])
            q, k = _turn(q, pos, freq, mag=mag), _turn(k, pos, freq, mag=mag)
            o = _each(seqs, lambda a, b: _attend(q[a:b], k[a:b], v[a:b], mx["scale"], "chunk", mx["mask"]["size"], w("mix.sink")))
            o = o.reshape(T, -1)
        elif kind == "gla":
            a_ = _mm(_mm(n, w("mix.a1")), w("mix.a2")) + w("mix.a2.b")
            decay = (torch.sigmoid(a_) ** (1.0 / mx["tau"])).view(T, H, D)
            o = _each(seqs, lambda a, b: _recurrence(q[a:b] / math.sqrt(D), k[a:b], v[a:b], decay[a:b]))
            o = (_unit(o, eps) * w("mix.norm")).reshape(T, -1) * _silu(_mm(n, w("mix.g")))
        else:
            decay = torch.tensor(mx["decay"], dtype=F64, device=DEVICE).view(1, H, 1).expand(T, H, D)
            q, k, v = _silu(q), _silu(k), _silu(v)
            o = _each(seqs, lambda a, b: _recurrence(q[a:b], k[a:b], v[a:b], decay[a:b]))
            o = _unit(o.reshape(T, -1), eps) * w("mix.norm") * torch.sigmoid(_mm(n, w("mix.g")))
        x = x + _mm(o, w("mix.o")) + _experts_exact(n, W, p + "mlp.", layer["mlp"], True)
        e = W["side.embed"][tok, i * side:(i + 1) * side].to(F64)
        x = x + _unit(_mm(_gelu(_mm(x, w("side.gate"))) * e, w("side.proj")), eps) * w("side.norm")
    return _mm(_unit(x[rows], eps) * W["final.norm"].to(F64), W["head"]) * cfg["logit_scale"]


def exact(case, seed):
    cfg, reqs, toks = _config(case), _requests(case), _tokens(case, seed)
    W = _weights(cfg, DTYPES[case["dtype"]], seed)
    tok = torch.tensor([t for one in toks for t in one], device=DEVICE)
    pos = torch.cat([torch.arange(len(t), device=DEVICE) for t in toks])
    seqs, at = [], 0
    for t in toks:
        seqs.append((at, at + len(t)))
        at += len(t)
    # the rows of the step's logits, then those of every further token
    sets = [[a + past + n - w + j for (a, _), (past, n, w) in zip(seqs, reqs) for j in range(w)]]
    sets += [[a + past + n + k for (a, _), (past, n, _) in zip(seqs, reqs)] for k in range(case["then"])]
    rows = torch.tensor([r for s in sets for r in s], device=DEVICE)
    forward = {"llama4": _llama4_exact, "ravenex": _ravenex_exact, "tebalorn": _tebalorn_exact}[case["model"]]
    z = forward(cfg, W, tok, pos, seqs, rows)
    return z if case["mode"] == "step" else list(z.split([len(s) for s in sets]))
