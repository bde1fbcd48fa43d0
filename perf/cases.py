"""The cases the engine's speed is measured on, and what their outputs have to be.

A case is one piece of work as a program that holds a loaded engine asks for it: requests brought in, their prompts run
through ``Engine.step``, their tokens generated by ``Engine.decode``, or the whole of it through a ``Session``'s ``run_batch``.
``prepare`` hands out what such a program has before the call (the engine with its weights, which a process loads once and
keeps, and the requests' prompts, which come from the seed), ``run`` is one pass, and ``exact`` is the same model in plain
torch in 64 bits.

Sizes.  LFM2-350M, 1.2B and 2.6B are the sizes ``bench.py`` runs, with pages of 16 tokens; Makuzen and Fazezen are its two
sets of sizes for them (latent attention over one cached row a token and experts chosen by a table; a fading matrix state,
attention within runs and retention).

Weights.  Drawn once from a fixed seed, so that every sub-layer moves the stream by a share that a trained model's would
(inputs of unit size in, outputs scaled down with the depth) and the next token is as decided as a trained model's mostly
is: the embedding is a good part of the stream at its end, and the head holds it (LFM2, Fazezen: the tied table; Makuzen:
the table shifted by one).  So two correct implementations generate the same tokens, and the logits beside them show how
far off each is.
"""
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from gesso_amd import BatchRequest, Engine, Sampler, Session, StepEntry, run_batch

DEVICE = "cuda:0"
VOCAB = 65536

# hidden, layers, heads, attention layers, feed-forward width (8 key heads, heads of 64, convolutions of 3 taps)
LFM2 = {
    "lfm2-350m": (1024, 16, 16, (2, 5, 8, 10, 12, 14), 4608),
    "lfm2-1.2b": (2048, 16, 32, (2, 5, 8, 10, 12, 14), 8192),
    "lfm2-2.6b": (2048, 30, 32, (2, 6, 10, 14, 18, 21, 24, 27), 7168),
}
KV_HEADS, HEAD, THETA = 8, 64, 1e6
# width, heads, plain / rotated / value width of a head, query and key/value rank, window, experts, used, widths (8 layers)
MAKUZEN = {
    "makuzen-1024": (1024, 16, 64, 32, 64, 384, 256, 1024, 16, 2, 512, 1024),
    "makuzen-2048": (2048, 16, 128, 64, 128, 768, 512, 2048, 32, 4, 704, 1408),
}
# width, head width of the fading state, heads and key heads of attention, runs, retention heads, feed-forward (8 layers)
FAZEZEN = {
    "fazezen-1024": (1024, 64, 16, 4, 512, 8, 4608),
    "fazezen-2048": (2048, 128, 32, 8, 1024, 16, 8192),
}
EPS = 1e-5


# ---------------------------------------------------------------------------- the cases

def _generate(model, batch, prompt, new, ragged=True, dtype="bfloat16", temperature=0.0, top_p=1.0, portion=2048, name=None):
    c = {"kind": "generate", "model": model, "dtype": dtype, "batch": batch, "prompt": prompt, "ragged": ragged, "new": new,
         "temperature": temperature, "top_p": top_p, "portion": portion}
    return dict(c, name=name) if name else c


def _prompt(model, tokens, every, dtype="bfloat16", name=None):
    c = {"kind": "prompt", "model": model, "dtype": dtype, "tokens": tokens, "every": every}
    return dict(c, name=name) if name else c


def _serve(model, requests, prompt, new, name=None):
    c = {"kind": "serve", "model": model, "dtype": "bfloat16", "requests": requests, "prompt": prompt, "new": new}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a short question to a small model: every launch and round trip counts
        _generate("lfm2-350m", 1, 13, 8, ragged=False, name="one-short-question"),
        # one user of the 1.2B sizes: decoding at batch 1
        _generate("lfm2-1.2b", 1, 512, 32, ragged=False, name="one-user"),
        # the benchmark's batch of 8 with 512-token prompts, lengths as they come
        _generate("lfm2-1.2b", 8, 512, 64, name="eight-users"),
        # a busy server: the most requests the fused decode loop takes
        _generate("lfm2-1.2b", 64, 200, 64, name="sixty-four-users"),
        # more requests than that, drawing from a nucleus: the decode loop over the many-row products
        _generate("lfm2-350m", 150, 100, 32, temperature=0.7, top_p=0.9, name="hundred-and-fifty-draws"),
        # the headline prompt
        _prompt("lfm2-1.2b", 2048, False, name="prompt-2048"),
        # a text of odd length scored: the logits of every position
        _prompt("lfm2-350m", 333, True, name="score-333"),
        # two long documents read in portions, then summed up
        _generate("lfm2-2.6b", 2, 16000, 32, name="long-documents"),
        # a session's own loop: requests of all lengths, portions of 512 beside decoding, half of the requests drawing
        _serve("lfm2-350m", 24, 1024, 96, name="session"),
        # the 32-bit path, as parity checks and careful users run it
        _generate("lfm2-1.2b", 6, 150, 16, dtype="float32", name="float32"),
        # the second architecture: latent rows and routed experts
        _generate("makuzen-2048", 8, 256, 32, name="makuzen"),
        # the third: matrix states beside attention within runs
        _generate("fazezen-2048", 8, 256, 32, name="fazezen"),
    ]


def _spread(rng, lo, hi):
    """A whole number, even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the same kinds over the same ranges (a drawn case needs no more work than the largest listed)."""
    top = max(_size(c) for c in listed())
    while True:
        kind = rng.choice(["few", "few", "many", "prompt", "prompt", "long", "serve", "float32", "other"])
        draws = rng.random() < 0.3
        t, p = (round(rng.uniform(0.5, 1.0), 2), round(rng.uniform(0.8, 1.0), 2)) if draws else (0.0, 1.0)
        if kind == "few":
            c = _generate(rng.choice(["lfm2-350m", "lfm2-1.2b"]), _spread(rng, 1, 64), _spread(rng, 8, 1024),
                          _spread(rng, 8, 64), True, "bfloat16", t, p)
        elif kind == "many":
            c = _generate("lfm2-350m", _spread(rng, 65, 256), _spread(rng, 16, 200), _spread(rng, 8, 32), True, "bfloat16", t, p)
        elif kind == "prompt":
            every = rng.random() < 0.4
            c = _prompt(rng.choice(sorted(LFM2)), _spread(rng, 16, 700 if every else 4096), every)
        elif kind == "long":
            c = _generate("lfm2-2.6b", rng.randint(1, 2), _spread(rng, 4000, 16000), _spread(rng, 8, 32))
        elif kind == "serve":
            c = _serve("lfm2-350m", rng.randint(6, 24), _spread(rng, 100, 1024), _spread(rng, 16, 96))
        elif kind == "float32":
            c = (_prompt(rng.choice(["lfm2-350m", "lfm2-1.2b"]), _spread(rng, 16, 1024), False, "float32") if rng.random() < 0.4 else
                 _generate(rng.choice(["lfm2-350m", "lfm2-1.2b"]), _spread(rng, 1, 8), _spread(rng, 16, 200), _spread(rng, 8, 16),
                           True, "float32"))
        else:
            c = _generate(rng.choice(sorted(MAKUZEN) + sorted(FAZEZEN)), _spread(rng, 1, 32), _spread(rng, 16, 512), _spread(rng, 8, 32),
                          True, "bfloat16", t, p)
        if _size(c) <= top:
            return c


# ---------------------------------------------------------------------------- models: configurations and weights

def _config(model, positions):
    if model in LFM2:
        from gesso_amd.config import Lfm2Config
        hidden, layers, heads, attn, ff = LFM2[model]
        return Lfm2Config.from_dict({
            "architectures": ["Lfm2ForCausalLM"], "vocab_size": VOCAB, "hidden_size": hidden, "num_hidden_layers": layers,
            "num_attention_heads": heads, "num_key_value_heads": KV_HEADS, "full_attn_idxs": list(attn), "conv_L_cache": 3,
            "conv_bias": False, "block_ff_dim": ff, "block_auto_adjust_ff_dim": False, "block_multiple_of": 256,
            "block_ffn_dim_multiplier": 1.0, "norm_eps": EPS, "rope_theta": THETA, "tie_word_embeddings": True,
            "max_position_embeddings": positions})
    if model in MAKUZEN:
        from gesso_amd.config import LatentAttentionConfig, MakuzenConfig, MakuzenLayer, TableMoEConfig, YarnScaling
        width, heads, dim, rot, vdim, qr, kr, window, experts, used, ff, shared = MAKUZEN[model]
        mixer = LatentAttentionConfig(heads=heads, dim=dim, rot_dim=rot, vdim=vdim, q_rank=qr, kv_rank=kr,
                                      scale=(dim + rot) ** -0.5, rot_base=THETA, scaling=YarnScaling(4.0, 1024.0, 32.0, 1.0),
                                      window=window)
        mlp = TableMoEConfig(experts=experts, top=used, ff=ff, shared_ff=shared)
        return MakuzenConfig(vocab=VOCAB, width=width, layers=tuple(MakuzenLayer(mixer, mlp) for _ in range(8)), embedding_scale=1.0,
                             norm_eps=EPS, residual_mult=0.5, max_position=positions)
    from gesso_amd.config import (ChunkedAttentionConfig, DenseConfig, FazezenConfig, FazezenLayer, LightningConfig,
                                  ParallelConfig, RetentionConfig, Rotation, Stretch)
    width, dim, heads, kv_heads, run, rheads, ff = FAZEZEN[model]
    light = FazezenLayer("lightning", LightningConfig(16, dim, dim, tuple(_fading())), DenseConfig(ff))
    pair = FazezenLayer("parallel", ParallelConfig(
        ChunkedAttentionConfig(heads, kv_heads, HEAD, HEAD, HEAD ** -0.5, Rotation(THETA, HEAD, Stretch(4.0, 1.0, 4.0, 2048.0)), run),
        RetentionConfig(rheads, 64, 128, tuple(_retained(rheads)), Rotation(THETA, 64)), 1.2, 0.9), DenseConfig(ff))
    return FazezenConfig(vocab=VOCAB, width=width, layers=tuple(pair if i in (2, 5) else light for i in range(8)), norm_eps=EPS,
                         max_position=positions)


def _fading():
    return [1.0 - 2.0 ** (-3 - 6 * h / 15) for h in range(16)]


def _retained(heads):
    return [1.0 - 2.0 ** (-5 - 5 * h / (heads - 1)) for h in range(heads)]


def _tables(model, positions):
    """The model as data, and its tensors' table: name -> shape and role."""
    from gesso_amd.config.registry import architecture_of
    from gesso_amd.models.model import tensor_table
    cfg = _config(model, positions)
    spec = architecture_of(cfg.to_json()).to_spec(cfg)
    return cfg, spec, tensor_table(spec)


def _weights(model, dtype, table):
    """Name -> tensor on the device, in the types a loader holds them in: matrices in ``dtype``, vectors in 32 bits."""
    gen = torch.Generator(device=DEVICE).manual_seed(20240131)
    wide = torch.float32 if dtype == "float32" else torch.bfloat16

    def normal(shape, std, mean=0.0):
        return torch.empty(tuple(shape), dtype=torch.float32, device=DEVICE).normal_(mean, std, generator=gen)

    out = {}
    for name, ts in table.items():
        shape, last = tuple(ts.shape), name.split(".")[-1]
        if ts.role == "index":                               # a row: different experts
            out[name] = torch.rand((shape[0], ts.high), device=DEVICE, generator=gen).argsort(dim=1)[:, :shape[1]].to(torch.int32)
            continue
        if ts.role == "vector":
            if name.endswith("conv.conv.weight"):
                t = normal(shape, 0.6)
            elif name.endswith("_layernorm.weight"):         # scores as spread as a trained model's: a few keys count
                t = normal(shape, 0.1, 1.5)
            else:
                t = normal(shape, 0.1, 1.0 if ts.init == "one_plus_normal" else 0.0)
            out[name] = t
            continue
        if name in ("model.embed_tokens.weight", "embed"):
            t = normal(shape, 1.0 if model in MAKUZEN else 0.05)
        elif name == "head":                                 # the token after v is v + 1
            t = 0.05 * out["embed"].float().roll(1, 0)
        else:
            std = shape[-1] ** -0.5
            if model in LFM2 and ("out_proj" in name or "w2" in name):
                std *= 0.02 * (16 / LFM2[model][1]) ** 0.5
            elif model in FAZEZEN and last in ("o", "down"):
                std *= 0.6
            t = normal(shape, std)
        out[name] = t.to(wide)
    return out


# ---------------------------------------------------------------------------- prepare and run

_held = {}           # the engine of the case at hand: a process loads its model once and keeps it


def _prompts(case, seed):
    rng = np.random.default_rng([seed, 7])
    kind = case["kind"]
    if kind == "prompt":
        lengths = [case["tokens"]]
    elif kind == "serve":
        lengths = [64] + np.exp(rng.uniform(math.log(64), math.log(case["prompt"]), case["requests"] - 1)).astype(int).tolist()
    elif case["ragged"]:
        lo = max(1, case["prompt"] // 2)
        lengths = rng.integers(lo, case["prompt"] + 1, case["batch"]).tolist()
        lengths[0] = case["prompt"]
    else:
        lengths = [case["prompt"]] * case["batch"]
    return [rng.integers(0, VOCAB, n).tolist() for n in lengths]


def _news(case):
    """How many tokens each request of a session asks for: the first the fewest, the last the most."""
    n = case["requests"]
    return [max(4, case["new"] * (i + 1) // n) for i in range(n)]


def _context(case):
    longest = case["tokens"] if case["kind"] == "prompt" else case["prompt"] + case["new"] + 1
    return max(4096, -(-longest // 1024) * 1024)


def _handle(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _held:
        _held.clear()
        torch.cuda.empty_cache()
        positions = _context(case)
        cfg, spec, table = _tables(case["model"], positions)
        tensors = _weights(case["model"], case["dtype"], table)
        if case["kind"] == "serve":
            _held[key] = _session(cfg, tensors, case)
        else:
            n = case.get("batch", 1)
            most = n * ((case["tokens"] if case["kind"] == "prompt" else case["prompt"] + case["new"]) + 32)
            _held[key] = Engine(spec, tensors, case["dtype"], DEVICE, page_size=16, max_tokens=most, num_slots=n + 1, max_context=positions)
    return _held[key]


def _session(cfg, tensors, case):
    """A session from a model folder, as a user starts one."""
    import json

    from gesso_amd.weights.safetensors_io import write_safetensors
    folder = tempfile.mkdtemp(prefix="model_")
    try:
        with open(os.path.join(folder, "config.json"), "w") as f:
            json.dump(cfg.to_json(), f)
        write_safetensors(os.path.join(folder, "model.safetensors"), {k: t.cpu() for k, t in tensors.items()})
        return Session(folder, dtype=case["dtype"], device=DEVICE, context_length=4096, max_num_seqs=64, chunk_size=512,
                       max_num_batched_tokens=2048, max_tokens=case["requests"] * (case["prompt"] + case["new"] + 32))
    finally:
        shutil.rmtree(folder)


def prepare(case, seed):
    return {"case": case, "seed": seed, "handle": _handle(case), "prompts": _prompts(case, seed)}


def _samplers(case, seed, n):
    if case["temperature"] <= 0:
        return None
    return [Sampler(case["temperature"], case["top_p"], seed + i) for i in range(n)]


def run(state):
    case, prompts = state["case"], state["prompts"]
    if case["kind"] == "serve":
        return _run_session(state["handle"], case, prompts, state["seed"])
    engine = state["handle"]
    if case["kind"] == "prompt":
        engine.add_request("p")
        try:
            n = len(prompts[0])
            return engine.step([StepEntry("p", prompts[0], list(range(n)) if case["every"] else [n - 1])])
        finally:
            engine.finish_request("p")
    rids = list(range(len(prompts)))
    for rid in rids:
        engine.add_request(rid)
    try:
        first = _read_prompts(engine, rids, prompts, case["portion"])
        tokens = first.argmax(1).tolist()
        samplers = _samplers(case, state["seed"], len(rids))
        ids, left = [], case["new"]
        while left:
            n = min(left, 32)
            got, _ = engine.decode(rids, tokens, n, samplers)
            ids.append(got)
            tokens = got[-1].tolist()
            left -= n
        last = engine.step([StepEntry(rid, [t], [0]) for rid, t in zip(rids, tokens)])
        return {"first": first, "tokens": np.concatenate(ids), "last": last}
    finally:
        for rid in rids:
            engine.finish_request(rid)


def _read_prompts(engine, rids, prompts, portion, budget=8192):
    """All prompts through steps of at most ``budget`` tokens, a request's portions of at most ``portion``: the logits of
    each prompt's last token."""
    done, rows = [0] * len(rids), [None] * len(rids)
    while any(d < len(p) for d, p in zip(done, prompts)):
        entries, ends, room = [], [], budget
        for i, (rid, p) in enumerate(zip(rids, prompts)):
            n = min(len(p) - done[i], portion, room)
            if n < 1:
                continue
            end = done[i] + n == len(p)
            entries.append(StepEntry(rid, p[done[i]:done[i] + n], [n - 1] if end else []))
            done[i] += n
            room -= n
            if end:
                ends.append(i)
        logits = engine.step(entries)
        for k, i in enumerate(ends):
            rows[i] = logits[k]
    return torch.stack(rows)


def _run_session(session, case, prompts, seed):
    """All requests together, each to its own length, every second one drawing; then the first text is scored."""
    requests = [BatchRequest(session, p, n, Sampler(0.7, 0.9, seed + i) if i % 2 else None)
                for i, (p, n) in enumerate(zip(prompts, _news(case)))]
    texts = [r.ids for r in run_batch(requests)]
    return {"tokens": _padded([t[len(p):] for t, p in zip(texts, prompts)], max(_news(case))), "score": session.prefill(texts[0])}


def _padded(rows, width):
    out = np.full((len(rows), width), -1, dtype=np.int64)
    for i, r in enumerate(rows):
        out[i, :len(r)] = r
    return out


# ---------------------------------------------------------------------------- what a pass cannot do without

def _params(model):
    """Weights a token's pass multiplies with (without the head), bytes and products a cached token costs."""
    if model in LFM2:
        H, L, nh, attn, F = LFM2[model]
        a = len(attn)
        return ((L - a) * 4 * H * H + a * (2 * nh * HEAD * H + 2 * KV_HEADS * HEAD * H) + L * 3 * H * F, H,
                a * 2 * KV_HEADS * HEAD, a * 2 * nh * HEAD, (L - a) * H * 2)
    if model in MAKUZEN:
        H, nh, n, r, v, qr, kr, window, experts, used, ff, shared = MAKUZEN[model]
        per = H * (qr + kr + r + nh) + qr * nh * (n + r) + kr * nh * (n + v) + nh * v * H + 2 * H * (used * ff + shared)
        return 8 * per, H, 8 * (kr + r), 8 * nh * (n + r + v), 0
    H, d, nh, nkv, run, rh, F = FAZEZEN[model]
    light, pair = 5 * H * 16 * d, H * (2 * nh * HEAD + 2 * nkv * HEAD) + H * (2 * rh * 64 + 3 * rh * 128)
    return (6 * light + 2 * pair + 8 * 3 * H * F, H, 2 * 2 * nkv * HEAD, 2 * 2 * nh * HEAD,
            6 * 16 * d * d + 2 * rh * 64 * 128)


def _expert_bytes(model, tokens):
    """Weights read by ``tokens`` tokens together: of routed experts those that some token uses."""
    params, H = _params(model)[:2]
    if model not in MAKUZEN:
        return params
    experts, used, ff = MAKUZEN[model][8:11]
    met = experts * (1 - (1 - used / experts) ** tokens)
    return params + 8 * 2 * H * ff * (met - used)


def work(case):
    model, width = case["model"], 4 if case["dtype"] == "float32" else 2
    params, H, kv, pair, state = _params(model)
    if case["kind"] == "prompt":
        T = case["tokens"]
        rows = T if case["every"] else 1
        return {"bytes": (params + VOCAB * H) * width + T * H * width + T * kv * width + rows * VOCAB * 4,
                "flops": 2.0 * (params * T + pair * T * (T + 1) / 2 + rows * VOCAB * H)}
    if case["kind"] == "serve":
        n, news = case["requests"], _news(case)
        mean = (case["prompt"] - 64) / math.log(case["prompt"] / 64) if case["prompt"] > 64 else 64.0
        lengths = [64.0] + [mean] * (n - 1)
    else:
        n, news = case["batch"], [case["new"]] * case["batch"]
        lengths = [float(case["prompt"])] + [case["prompt"] * (0.75 if case["ragged"] else 1.0)] * (n - 1)
    bytes_, flops = 0.0, 0.0
    tokens = sum(lengths)
    bytes_ += (_expert_bytes(model, tokens) + VOCAB * H) * width + tokens * (H + kv) * width
    flops += 2.0 * (params * tokens + sum(pair * t * t / 2 for t in lengths) + n * VOCAB * H)
    for s in range(max(news) + (case["kind"] == "generate")):       # (generate: one more step for the last logits)
        live = [t + s for t, w in zip(lengths, news) if s < w + (case["kind"] == "generate")]
        bytes_ += (_expert_bytes(model, len(live)) + VOCAB * H) * width + sum(live) * kv * width + len(live) * state * 8
        flops += 2.0 * (len(live) * (params + VOCAB * H) + pair * sum(live))
    bytes_ += 2 * n * VOCAB * 4
    return {"bytes": bytes_, "flops": flops}


def _size(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def tolerance(case):
    """Relative error of the logits; the tokens are the same.  Against ``exact`` the logits stand 0.9 to 1.1e-2 off in
    bfloat16 (LFM2; 7e-3 and 5e-3 for the other two) and 9e-7 in 32 bits; two implementations that round in other places
    differ by the root of twice the square."""
    if case["dtype"] == "float32":
        return {"rel": 5e-6, "max": 1e-4, "differ": 0.0}
    return {"rel": 3e-2 if case["model"] in LFM2 else 2e-2, "max": 2e-1, "differ": 0.0}


# ---------------------------------------------------------------------------- the same in 64 bits

def _rms(x, weight=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)
    return y if weight is None else y * weight


def _turned(x, freqs, mult=1.0, sign=1.0):
    """``x (T, heads, width)``, feature i of a head turned with feature i + len(freqs) by the position."""
    T, half = x.shape[0], len(freqs)
    a = torch.arange(T, dtype=torch.float64, device=DEVICE)[:, None] * torch.tensor(freqs, dtype=torch.float64, device=DEVICE)
    c, s = (a.cos() * mult)[:, None], (a.sin() * mult * sign)[:, None]
    u, v = x[..., :half], x[..., half:2 * half]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * half:]], -1)


def _freqs(dims):
    return [THETA ** (-2.0 * i / dims) for i in range(dims // 2)]


def _attention(q, k, v, scale, first, sink=False):
    """``q (T, H, n)``, ``k (T, H, n)``, ``v (T, H, m)``: softmax over the keys ``first(i) <= j <= i``; with ``sink`` one
    more term exp(0) in the denominator."""
    T, out = q.shape[0], []
    q, k, v = q.transpose(0, 1), k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous()
    j = torch.arange(T, device=DEVICE)
    for at in range(0, T, 512):
        i = torch.arange(at, min(at + 512, T), device=DEVICE)
        end = int(i[-1]) + 1
        s = torch.matmul(q[:, at:end], k[:, :end].transpose(1, 2).contiguous()) * scale
        s = s.masked_fill(~((j[None, :end] <= i[:, None]) & (j[None, :end] >= first(i)[:, None])), -math.inf)
        if sink:
            s = torch.cat([s, torch.zeros_like(s[..., :1])], -1)
        p = torch.softmax(s, -1)
        out.append(torch.matmul(p[..., :end], v[:, :end]))
    return torch.cat(out, 1).transpose(0, 1)


def _grouped(x, heads):
    return x.repeat_interleave(heads // x.shape[1], 1)


def _lfm2_layer(model, w, i, x, cuts):
    H, L, nh, attn, F = LFM2[model]
    p = f"model.layers.{i}."
    h = _rms(x, w(p + "operator_norm.weight"))
    if i in attn:
        q = (h @ w(p + "self_attn.q_proj.weight").t()).view(-1, nh, HEAD)
        k = (h @ w(p + "self_attn.k_proj.weight").t()).view(-1, KV_HEADS, HEAD)
        v = (h @ w(p + "self_attn.v_proj.weight").t()).view(-1, KV_HEADS, HEAD)
        q, k = _rms(q, w(p + "self_attn.q_layernorm.weight")), _rms(k, w(p + "self_attn.k_layernorm.weight"))
        f = _freqs(HEAD)
        y = torch.cat([_attention(_turned(q[a:b], f), _grouped(_turned(k[a:b], f), nh), _grouped(v[a:b], nh), HEAD ** -0.5,
                                  lambda i: torch.zeros_like(i)) for a, b in cuts]).reshape(len(x), -1)
        y = y @ w(p + "self_attn.out_proj.weight").t()
    else:
        b, c, u = (h @ w(p + "conv.in_proj.weight").t()).chunk(3, 1)
        z, taps = b * u, w(p + "conv.conv.weight").view(H, 3)
        y = torch.zeros_like(z)
        for lo, hi in cuts:
            for t in range(3):                               # tap t is for the token 2 - t places back
                y[lo + 2 - t:hi] += z[lo:hi - 2 + t] * taps[:, t] if hi - lo > 2 - t else 0.0
        y = (c * y) @ w(p + "conv.out_proj.weight").t()
    x = x + y
    h = _rms(x, w(p + "ffn_norm.weight"))
    g = torch.nn.functional.silu(h @ w(p + "feed_forward.w1.weight").t()) * (h @ w(p + "feed_forward.w3.weight").t())
    return x + g @ w(p + "feed_forward.w2.weight").t()


def _yarn(dims, factor=4.0, original=1024.0, fast=32.0, slow=1.0):
    def dim_of(turns):
        return dims * math.log(original / (2 * math.pi * turns)) / (2 * math.log(THETA))
    lo, hi = max(math.floor(dim_of(fast)), 0), min(math.ceil(dim_of(slow)), dims - 1)
    out = []
    for i, f in enumerate(_freqs(dims)):
        r = min(1.0, max(0.0, (i - lo) / max(hi - lo, 0.001)))
        out.append(f / factor * r + f * (1 - r))
    return out, 0.1 * math.log(factor) + 1.0


def _makuzen_layer(model, w, i, x, cuts, ids):
    H, nh, n, r, vd, qr, kr, window, experts, used, ff, shared = MAKUZEN[model]
    p, T = f"l{i}.mix.", len(x)
    freqs, mult = _yarn(r)
    q = (_rms(x @ w(p + "dq").t(), w(p + "dq.norm")) @ w(p + "uq").t()).view(T, nh, n + r)
    down = x @ w(p + "dkv").t()
    z = _rms(down[:, :kr], w(p + "dkv.norm"))
    k, v = (z @ w(p + "uk").t()).view(T, nh, n), (z @ w(p + "uv").t()).view(T, nh, vd)
    out = []
    for a, b in cuts:
        qr_, kr_ = _turned(q[a:b, :, n:], freqs, mult), _turned(down[a:b, None, kr:], freqs, mult)
        out.append(_attention(torch.cat([q[a:b, :, :n], qr_], -1), torch.cat([k[a:b], kr_.expand(-1, nh, -1)], -1), v[a:b],
                              (n + r) ** -0.5, lambda i: (i - window + 1).clamp(min=0)))
    y = torch.cat(out) * torch.sigmoid(x @ w(p + "g").t())[:, :, None]
    x = x + 0.5 * _rms(y.reshape(T, -1) @ w(p + "o").t(), w(f"l{i}.norm1"))
    p = f"l{i}.mlp."
    chosen, y = w(p + "table")[ids], torch.zeros_like(x)
    for e in range(experts):
        at = (chosen == e).any(1).nonzero()[:, 0]
        if len(at):
            y[at] += torch.relu(x[at] @ w(f"{p}e{e}.up").t()).square() @ w(f"{p}e{e}.down").t() / used
    y += torch.sigmoid(x @ w(p + "shared.sg").view(-1, 1)) * (torch.relu(x @ w(p + "shared.up").t()).square() @ w(p + "shared.down").t())
    return x + 0.5 * _rms(y, w(f"l{i}.norm2"))


def _faded(q, k, v, decay):
    """``o_t = sum over s <= t of d^(t - s) (q_t . k_s) v_s`` per head."""
    T = q.shape[0]
    t = torch.arange(T, dtype=torch.float64, device=DEVICE)
    gap = t[:, None] - t[None]
    out = []
    for h, d in enumerate(decay):
        s = (q[:, h] @ k[:, h].t()) * torch.where(gap >= 0, torch.exp(gap * math.log(d)), 0.0)
        out.append(s @ v[:, h])
    return torch.stack(out, 1)


def _stretched(factor=4.0, low=1.0, high=4.0, original=2048.0):
    out = []
    for f in _freqs(HEAD):
        s = (original * f / (2 * math.pi) - low) / (high - low)
        out.append(f if s > 1 else f / factor if s < 0 else (1 - s) * f / factor + s * f)
    return out


def _fazezen_layer(model, w, i, x, cuts):
    H, d, nh, nkv, run, rh, F = FAZEZEN[model]
    p, T, silu = f"l{i}.mix.", len(x), torch.nn.functional.silu
    h = _rms(x, 1 + w(f"l{i}.norm1"))
    if i not in (2, 5):
        q, k, v = (silu(h @ w(p + n).t()).view(T, 16, d) for n in "qkv")
        o = torch.cat([_faded(q[a:b], k[a:b], v[a:b], _fading()) for a, b in cuts]).reshape(T, -1)
        y = (_rms(o, w(p + "norm")) * torch.sigmoid(h @ w(p + "g").t())) @ w(p + "o").t()
    else:
        l, f, plain = p + "left.", _stretched(), _freqs(HEAD)
        q = _rms((h @ w(l + "q").t()).view(T, nh, HEAD), w(l + "q.norm"))
        k = _rms((h @ w(l + "k").t()).view(T, nkv, HEAD), w(l + "k.norm"))
        v = (h @ w(l + "v").t()).view(T, nkv, HEAD)
        o = torch.cat([_turned(_attention(_turned(q[a:b], f), _grouped(_turned(k[a:b], f), nh), _grouped(_turned(v[a:b], plain), nh),
                                          HEAD ** -0.5, lambda i: i // run * run, sink=True), plain, sign=-1.0) for a, b in cuts])
        y = 1.2 * (o.reshape(T, -1) @ w(l + "o").t())
        r = p + "right."
        q, k = ((h @ w(r + n).t()).view(T, rh, 64) for n in "qk")
        v, f = (h @ w(r + "v").t()).view(T, rh, 128), _freqs(64)
        o = torch.cat([_rms(_faded(_turned(q[a:b], f), _turned(k[a:b], f) / 8.0, v[a:b], _retained(rh))) for a, b in cuts])
        y = y + 0.9 * ((o.reshape(T, -1) * silu(h @ w(r + "g").t())) @ w(r + "o").t())
    p = f"l{i}.mlp."
    h = _rms(x, 1 + w(f"l{i}.norm2"))
    g = torch.nn.functional.gelu(h @ w(p + "gate").t() + w(p + "gate.b"), approximate="tanh") * (h @ w(p + "up").t() + w(p + "up.b"))
    return x + y + g @ w(p + "down").t() + w(p + "down.b")


def _logits(case, texts, froms):
    """Per text the logits ``(len - from, vocab)`` of its positions from ``from`` on."""
    model, (_, _, table) = case["model"], _tables(case["model"], _context(case))
    raw = _weights(model, case["dtype"], table)

    def w(name):
        t = raw[name]
        return t.double() if t.is_floating_point() else t.long()

    ids = torch.tensor([t for text in texts for t in text], device=DEVICE)
    ends = np.cumsum([len(t) for t in texts]).tolist()
    cuts = list(zip([0] + ends[:-1], ends))
    x = raw["model.embed_tokens.weight" if model in LFM2 else "embed"][ids].double()
    if model in FAZEZEN:
        x = _rms(x, 1 + w("embed.norm"))
    for i in range(LFM2[model][1] if model in LFM2 else 8):
        x = (_lfm2_layer(model, w, i, x, cuts) if model in LFM2 else _makuzen_layer(model, w, i, x, cuts, ids) if model in MAKUZEN
             else _fazezen_layer(model, w, i, x, cuts))
    keep = torch.cat([torch.arange(a + f, b, device=DEVICE) for (a, b), f in zip(cuts, froms)])
    x = x[keep]
    if model in LFM2:
        x, head = _rms(x, w("model.embedding_norm.weight")), "model.embed_tokens.weight"
    else:
        x, head = _rms(x, w("final.norm") if model in MAKUZEN else 1 + w("final.norm")), "head" if model in MAKUZEN else "embed"
    return (x @ w(head).t()).split([b - a - f for (a, b), f in zip(cuts, froms)])


def exact(case, seed):
    prompts = _prompts(case, seed)
    if case["kind"] == "prompt":
        return _logits(case, prompts, [0 if case["every"] else len(prompts[0]) - 1])[0]
    # what is generated if every step's best is the head's partner of the token before it, checked step by step below
    serve = case["kind"] == "serve"
    news = _news(case) if serve else [case["new"] + 1] * len(prompts)
    step = 1 if case["model"] in MAKUZEN else 0
    new = [[(p[-1] + step * (k + 1)) % VOCAB for k in range(n)] for p, n in zip(prompts, news)]
    texts = [p + t for p, t in zip(prompts, new)]
    rows = _logits(case, texts, [0 if serve and i == 0 else len(p) - 1 for i, p in enumerate(prompts)])
    sure = all(torch.equal(r[-n - 1:-1].argmax(1).cpu(), torch.tensor(t)) for r, t, n in zip(rows, new, news))
    if serve:
        return {"tokens": _padded(new, max(news)) if sure else None, "score": rows[0]}
    tokens = np.array(new).T[1:].astype(np.int32) if sure else None
    return {"first": torch.stack([r[0] for r in rows]), "tokens": tokens, "last": torch.stack([r[-1] for r in rows]) if sure else None}
