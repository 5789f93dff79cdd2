"""The work that a user of the engine has it do, as cases that can be timed and checked.

``listed()`` names them, ``draw(rng)`` gives more of the same ranges, ``prepare`` makes what a server holds before a step
(model, cache, requests under way), ``run`` is one pass through ``LLM.step_raw`` or ``Sampler.sample``, and ``exact`` is the
same pass in 64 bits, in plain torch and without this package's code.  Kinds of a pass:

``decode``    one step of a token a request, every request with a context of its own length behind it.  A pass leaves the
              contexts a token longer, as serving does.
``prompt``    one or several prompts from their first token to the logits of their last one, whole or in portions.
``mixed``     a decoding step that also takes in a whole short prompt: what chunked prefill makes of a busy server's steps.
``sampling``  the choice of every row's next token, rows with options of their own.

Models: ``qwen3-8b``, the shape of the benchmark, all 36 layers in bfloat16; ``qwen3-2k-float32``, four layers of width 2,048 in
the true 32-bit run; ``sosuvik-4k``, four layers of width 4,096 with attention in chunks, latent attention and grouped routed
experts, the newest of the other designs, whose routed experts, latent rows and capped attention the others share.
"""
from __future__ import annotations

import math
import zlib

import numpy as np
import torch

DEVICE = "cuda:0"
PAGE = 16
ROOM = 1536          # tokens that a decoding request can grow by before it starts over at its first length
F64 = torch.float64

QWEN = {
    "qwen3-8b": dict(vocab_size=151936, hidden_size=4096, intermediate_size=12288, num_hidden_layers=36,
                     num_attention_heads=32, num_key_value_heads=8),
    "qwen3-2k-float32": dict(vocab_size=32000, hidden_size=2048, intermediate_size=8192, num_hidden_layers=4,
                             num_attention_heads=16, num_key_value_heads=4),
}
QWEN_REST = dict(architectures=["Qwen3ForCausalLM"], head_dim=128, max_position_embeddings=40960, rms_norm_eps=1e-6,
                 rope_theta=1e6, tie_word_embeddings=False, torch_dtype="bfloat16", use_sliding_window=False)

_BLENDED = {"factor": 4.0, "original": 8192, "fast": 32.0, "slow": 1.0}
_ROUTED = {"expert": {"ff": 1536, "limit": 7.0}, "kind": "moe",
           "router": {"experts": 16, "groups": {"count": 4, "keep": 2}, "scale": 2.0, "top": 4}}
_CHUNKED = {"type": "attention", "mlp": _ROUTED,
            "mixer": {"dim": 128, "heads": 32, "kv_heads": 8, "mask": {"size": 1024}, "scale": 128 ** -0.5, "softcap": 30.0,
                      "rot": {"base": 1e6, "dims": 128, "scaling": _BLENDED}, "vdim": 128}}
_LATENT = {"type": "latent_attention", "mlp": _ROUTED,
           "mixer": {"dim": 128, "heads": 32, "kv_rank": 512, "rot": {"base": 1e6, "dims": 64}, "rot_dim": 64,
                     "scale": 192 ** -0.5, "vdim": 128}}
SOSUVIK = {"architecture": "Sosuvik", "vocab": 32000, "width": 4096, "norm": {"eps": 1e-6}, "logit_scale": 0.5,
           "loop": {"start": 0, "stop": 2, "times": 1}, "layers": [_CHUNKED, _LATENT, _CHUNKED, _LATENT]}


# ---------------------------------------------------------------------------------------------------- the cases
def listed():
    big = "qwen3-8b"
    return [
        # One user's chat: the step's latency is all there is.
        {"name": "decode-1", "model": big, "kind": "decode", "requests": 1, "shortest": 600, "longest": 600},
        # The headline benchmark: batch 8, contexts of about 4,096.
        {"name": "decode-8", "model": big, "kind": "decode", "requests": 8, "shortest": 3900, "longest": 3900},
        # A server's usual step: requests of all lengths, as the serving benchmark's prompts and answers make them.
        {"name": "decode-32-ragged", "model": big, "kind": "decode", "requests": 32, "shortest": 128, "longest": 1664},
        # A server that takes a prompt in while it decodes: more rows than a decoding step has, fewer than a prompt's.
        {"name": "mixed-24-and-333", "model": big, "kind": "mixed", "requests": 24, "shortest": 200, "longest": 1300,
         "tokens": 333},
        # A short question, an ordinary prompt of an odd length, the benchmark's prompt, a long document.
        {"name": "prompt-97", "model": big, "kind": "prompt", "prompts": 1, "tokens": 97, "portion": 0},
        {"name": "prompt-509", "model": big, "kind": "prompt", "prompts": 1, "tokens": 509, "portion": 0},
        {"name": "prompt-2048", "model": big, "kind": "prompt", "prompts": 1, "tokens": 2048, "portion": 0},
        {"name": "prompt-8192", "model": big, "kind": "prompt", "prompts": 1, "tokens": 8192, "portion": 0},
        # The 32-bit run (``--dtype float32``), by which users check a checkpoint.
        {"name": "float32-prompt-333", "model": "qwen3-2k-float32", "kind": "prompt", "prompts": 1, "tokens": 333, "portion": 0},
        # Another design's prompt and decoding step: routed experts, attention in chunks, latent attention.
        {"name": "sosuvik-prompt-2048", "model": "sosuvik-4k", "kind": "prompt", "prompts": 1, "tokens": 2048, "portion": 0},
        {"name": "sosuvik-decode-8", "model": "sosuvik-4k", "kind": "decode", "requests": 8, "shortest": 1500, "longest": 1500},
        # The tokens of a serving step: greedy rows, temperatures, top-k, top-p, presence penalties side by side.
        {"name": "sampling-32", "model": "none", "kind": "sampling", "rows": 32, "vocab": 151936},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "decode", "prompt", "prompt", "prompt", "mixed", "sampling"))
    if kind == "sampling":
        return {"model": "none", "kind": kind, "rows": _log_int(rng, 1, 64), "vocab": rng.choice((32000, 151936))}
    model = rng.choice(("qwen3-8b", "qwen3-8b", "sosuvik-4k", "qwen3-2k-float32" if kind == "prompt" else "qwen3-8b"))
    if kind == "prompt":
        most = 1024 if model == "qwen3-2k-float32" else 8192
        prompts = rng.choice((1, 1, 1, 2, 3, 4))
        tokens = _log_int(rng, 12, most // prompts)
        portion = rng.choice((0, 0, 512)) if tokens > 512 else 0
        return {"model": model, "kind": kind, "prompts": prompts, "tokens": tokens, "portion": portion}
    requests = _log_int(rng, 1, 64 if kind == "decode" else 32)
    most = min(8000, 32000 // requests)
    longest = _log_int(rng, 64, most)
    shortest = longest if rng.random() < 0.4 else rng.randint(16, longest)
    case = {"model": model, "kind": kind, "requests": requests, "shortest": shortest, "longest": longest}
    if kind == "mixed":
        case["tokens"] = _log_int(rng, 12, 512)
    return case


# ---------------------------------------------------------------------------------------------------- inputs from the seed
def _vocab(model):
    return QWEN[model]["vocab_size"] if model in QWEN else SOSUVIK["vocab"]


def _contexts(case):
    """The lengths of the contexts behind a decoding step's tokens."""
    n, low, high = case["requests"], case["shortest"], case["longest"]
    return [int(v) for v in np.random.default_rng(n * 7919 + high).integers(low, high + 1, n)] if low < high else [high] * n


def _traffic(case, seed):
    """Token ids: the contexts, the tokens that the decoding steps are given in turn, the prompts."""
    r = np.random.default_rng(seed)
    vocab = _vocab(case["model"])
    lengths = _contexts(case) if "requests" in case else []
    contexts = [r.integers(0, vocab, n).tolist() for n in lengths]
    steps = r.integers(0, vocab, (64, len(lengths))).tolist()
    prompts = [r.integers(0, vocab, case["tokens"]).tolist() for _ in range(case.get("prompts", 1))] if "tokens" in case else []
    return contexts, steps, prompts


class Checkpoint:
    """A checkpoint's tensors by name, each made from the seed and its name when it is asked for: matrices normal with
    standard deviation 1 / sqrt(inputs), norm weights 1 + U(-0.1, 0.1)."""

    origin = "<seeded>"

    def __init__(self, model, seed):
        self.model, self.seed = model, int(seed)
        self.shapes = qwen_shapes(QWEN[model]) if model in QWEN else sosuvik_shapes(SOSUVIK)

    def names(self):
        return list(self.shapes)

    def info(self, name):
        return torch.bfloat16, self.shapes[name]

    def generator(self, name):
        return torch.Generator(device=DEVICE).manual_seed((self.seed * 1000003 + zlib.crc32(name.encode())) & 0x7FFFFFFFFFFF)

    def get(self, name):
        shape, gen = self.shapes[name], self.generator(name)
        if self.model not in QWEN and (special := sosuvik_special(self, name, shape, gen)) is not None:
            return special.to(torch.bfloat16)
        if len(shape) == 1:
            return (torch.rand(shape, generator=gen, device=DEVICE) * 0.2 + 0.9).to(torch.bfloat16)
        std = 0.02 if "embed" in name else shape[1] ** -0.5
        return torch.empty(shape, dtype=torch.bfloat16, device=DEVICE).normal_(0.0, std, generator=gen)


def qwen_shapes(c):
    h, f, d = c["hidden_size"], c["intermediate_size"], QWEN_REST["head_dim"]
    nq, nkv = c["num_attention_heads"], c["num_key_value_heads"]
    out = {"model.embed_tokens.weight": (c["vocab_size"], h), "model.norm.weight": (h,), "lm_head.weight": (c["vocab_size"], h)}
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        out.update({p + "input_layernorm.weight": (h,), p + "post_attention_layernorm.weight": (h,),
                    p + "self_attn.q_proj.weight": (nq * d, h), p + "self_attn.k_proj.weight": (nkv * d, h),
                    p + "self_attn.v_proj.weight": (nkv * d, h), p + "self_attn.o_proj.weight": (h, nq * d),
                    p + "self_attn.q_norm.weight": (d,), p + "self_attn.k_norm.weight": (d,),
                    p + "mlp.gate_proj.weight": (f, h), p + "mlp.up_proj.weight": (f, h), p + "mlp.down_proj.weight": (h, f)})
    return out


def sosuvik_shapes(c):
    h, loop = c["width"], c["loop"]
    out = {"embed": (c["vocab"], h), "final.norm": (h,), "head": (c["vocab"], h), "loop.in": (h, 2 * h),
           "loop.step": (loop["times"], h)}
    for i, layer in enumerate(c["layers"]):
        p, m, e = f"l{i}.", layer["mixer"], layer["mlp"]
        out.update({p + "norm1": (h,), p + "norm2": (h,), p + "mix.o": (h, m["heads"] * m["vdim"])})
        if layer["type"] == "attention":
            out.update({p + "mix.q": (m["heads"] * m["dim"], h), p + "mix.k": (m["kv_heads"] * m["dim"], h),
                        p + "mix.v": (m["kv_heads"] * m["vdim"], h)})
        else:
            out.update({p + "mix.q": (m["heads"] * (m["dim"] + m["rot_dim"]), h), p + "mix.dkv": (m["kv_rank"] + m["rot_dim"], h),
                        p + "mix.dkv.norm": (m["kv_rank"],), p + "mix.uk": (m["heads"] * m["dim"], m["kv_rank"]),
                        p + "mix.uv": (m["heads"] * m["vdim"], m["kv_rank"])})
        n, ff = e["router"]["experts"], e["expert"]["ff"]
        out.update({p + "mlp.router": (n, h), p + "mlp.correction": (n,)})
        for j in range(n):
            out.update({p + f"mlp.e{j}.gate": (ff, h), p + f"mlp.e{j}.up": (ff, h), p + f"mlp.e{j}.down": (h, ff)})
    return out


def sosuvik_special(source, name, shape, gen):
    """What a trained model has and random weights lack: a router that is sure.  Every token has two groups and two experts of
    each, its embedding has a part in these experts' directions, the routers look for the directions, and the product that
    brings the embedding back in keeps them.  (With routers at chance a rounded bit somewhere sends a token elsewhere.)"""
    if name == "embed" or name.endswith("mlp.router"):
        r = _ROUTED["router"]
        experts, groups, keep, top = r["experts"], r["groups"]["count"], r["groups"]["keep"], r["top"]
        along = torch.randn((experts, shape[1]), generator=source.generator("directions"), device=DEVICE).sign() * shape[1] ** -0.5
        if name != "embed":
            return 0.15 * along
        kept = torch.rand((shape[0], groups), generator=gen, device=DEVICE).argsort(1)[:, :keep]
        size, each = experts // groups, top // keep
        inside = torch.rand((shape[0], keep, size), generator=gen, device=DEVICE).argsort(2)[:, :, :each]
        chosen = torch.zeros((shape[0], experts), device=DEVICE).scatter_(1, (kept.unsqueeze(2) * size + inside).flatten(1), 16.0)
        return torch.randn(shape, generator=gen, device=DEVICE) + chosen @ along
    if name.endswith("mlp.correction"):
        return torch.rand(shape, generator=gen, device=DEVICE) * 0.04 - 0.02
    if name == "loop.in":
        half = 0.5 * torch.eye(shape[0], device=DEVICE)
        return torch.cat([half, half], dim=1) + 0.1 * shape[1] ** -0.5 * torch.randn(shape, generator=gen, device=DEVICE)
    if name == "loop.step":
        return 0.1 * torch.randn(shape, generator=gen, device=DEVICE)
    return None


def _llm(case, seed, requests, tokens):
    from pulse_infer_amd import LLM, Qwen3Config, SosuvikConfig
    from pulse_infer_amd.models.factory import build_model

    model = case["model"]
    cfg = Qwen3Config.from_dict(dict(QWEN_REST, **QWEN[model]), "<cases>") if model in QWEN \
        else SosuvikConfig.from_dict(SOSUVIK, "<cases>")
    built = build_model(cfg, Checkpoint(model, seed), mode="float32" if model.endswith("float32") else "bfloat16", device=DEVICE)
    pages = sum((n + PAGE - 1) // PAGE + 1 for n in tokens)
    return LLM(built, cfg, max_batch_size=requests, page_size=PAGE, num_pages=pages, max_sequences=requests)


SAMPLING = (dict(), dict(temperature=0.7), dict(temperature=0.8, top_p=0.9), dict(temperature=1.0, top_k=50),
            dict(temperature=0.7, top_k=200, top_p=0.95, presence_penalty=1.5))


def prepare(case, seed):
    if case["kind"] == "sampling":
        from pulse_infer_amd import SamplingParams
        from pulse_infer_amd.sampling.sampler import Sampler

        rows, vocab = case["rows"], case["vocab"]
        gen = torch.Generator(device=DEVICE).manual_seed(seed)
        logits = torch.randn((rows, vocab), generator=gen, device=DEVICE) * 3.0
        params = [SamplingParams(seed=seed * 64 + i, **SAMPLING[i % len(SAMPLING)]) for i in range(rows)]
        sampler = Sampler(vocab, rows, torch.device(DEVICE))
        r = np.random.default_rng(seed)
        for i, p in enumerate(params):
            sampler.start_request(i, p, r.integers(0, vocab, 200).tolist())
        return {"kind": "sampling", "sampler": sampler, "logits": logits, "params": params}
    contexts, steps, prompts = _traffic(case, seed)
    llm = _llm(case, seed, len(contexts) + len(prompts), [len(c) + ROOM for c in contexts] + [len(p) for p in prompts])
    state = {"kind": case["kind"], "llm": llm, "lengths": [len(c) for c in contexts], "steps": steps, "prompts": prompts,
             "portion": case.get("portion", 0), "done": 0}
    # the requests under way: their contexts computed by the model, a few thousand tokens a step
    batch = []
    for i, c in enumerate(contexts):
        batch.append({"id": i, "tokens": c})
        if i + 1 == len(contexts) or sum(len(e["tokens"]) for e in batch) + len(contexts[i + 1]) > 4096:
            llm.step_raw(batch)
            batch = []
    return state


# ---------------------------------------------------------------------------------------------------- one pass
def run(state):
    if state["kind"] == "sampling":
        rows = len(state["params"])
        return np.array(state["sampler"].sample(state["logits"], state["params"], range(rows), [17] * rows, [0] * rows))
    llm, prompts = state["llm"], state["prompts"]
    if state["kind"] == "prompt":
        n = len(prompts[0])
        step = state["portion"] or n
        for at in range(0, n, step):
            last = at + step >= n
            entries = [{"id": f"p{i}", "tokens": p[at:at + step], "want": [len(p[at:at + step]) - 1] if last else []}
                       for i, p in enumerate(prompts)]
            logits = llm.step_raw(entries, end=[e["id"] for e in entries] if last else ())
        return logits
    if state["done"] == ROOM:      # the requests have grown as far as their pages go: they start over
        runner = llm.engine.runner
        for i in range(len(state["lengths"])):
            runner.free_request(("raw", i))
        for i, n in enumerate(state["lengths"]):
            runner.add_request(("raw", i))
            runner.reserve(("raw", i), n)
            runner.cache.advance(("raw", i), n)
        state["done"] = 0
    tokens = state["steps"][state["done"] % len(state["steps"])]
    state["done"] += 1
    entries = [{"id": i, "tokens": [t], "want": [0]} for i, t in enumerate(tokens)]
    entries += [{"id": "new", "tokens": p, "want": [len(p) - 1]} for p in prompts]
    return llm.step_raw(entries, end=["new"] if prompts else ())


# ---------------------------------------------------------------------------------------------------- what a pass cannot do without
def _sequences(case):
    """(tokens before the pass, tokens of the pass) of every request."""
    out = [(n, 1) for n in _contexts(case)] if "requests" in case else []
    return out + [(0, case["tokens"])] * case.get("prompts", 1) if "tokens" in case else out


def _in_chunks(before, n, size):
    """The same, cut where a chunk of ``size`` positions ends: (tokens of the chunk before, tokens of the pass in it)."""
    return [(max(before, t) - t, min(before + n, t + size) - max(before, t)) for t in range(before // size * size, before + n, size)]


def work(case):
    if case["kind"] == "sampling":
        n = case["rows"] * case["vocab"]
        return {"bytes": 4.0 * n, "flops": 2.0 * n}
    seqs = _sequences(case)
    tokens, wanted = sum(n for _, n in seqs), len(seqs)
    size = 4 if case["model"].endswith("float32") else 2
    pairs = lambda before, n: n * before + n * (n + 1) / 2.0
    if case["model"] in QWEN:
        c, d = QWEN[case["model"]], QWEN_REST["head_dim"]
        h, f, nq, nkv, layers, vocab = (c["hidden_size"], c["intermediate_size"], c["num_attention_heads"],
                                        c["num_key_value_heads"], c["num_hidden_layers"], c["vocab_size"])
        weights = layers * (h * (2 * nq + 2 * nkv) * d + 3 * h * f)
        cache = layers * 2 * nkv * d * sum(b + n for b, n in seqs)
        flops = 2.0 * weights * tokens + layers * 4.0 * nq * d * sum(pairs(b, n) for b, n in seqs)
        read = weights
    else:
        h, vocab = SOSUVIK["width"], SOSUVIK["vocab"]
        read, cache, flops = 2 * h * h, 0.0, 2.0 * 2 * h * h * tokens
        for layer in SOSUVIK["layers"]:
            m, r = layer["mixer"], layer["mlp"]["router"]
            expert, used = 3 * h * layer["mlp"]["expert"]["ff"], r["experts"] * (1 - (1 - r["top"] / r["experts"]) ** tokens)
            if layer["type"] == "attention":
                mix, size_c = h * (2 * m["heads"] + 2 * m["kv_heads"]) * m["dim"], m["mask"]["size"]
                begun = [part for b, n in seqs for part in _in_chunks(b, n, size_c)]
                flops += 4.0 * m["heads"] * m["dim"] * sum(pairs(b, n) for b, n in begun)
                cache += 2 * m["kv_heads"] * m["dim"] * sum(b + n for b, n in begun)
            else:
                mix = h * (m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]) + m["kv_rank"] + m["rot_dim"]) \
                    + m["kv_rank"] * m["heads"] * (m["dim"] + m["vdim"])
                flops += 2.0 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]) * sum(pairs(b, n) for b, n in seqs)
                cache += (m["kv_rank"] + m["rot_dim"]) * sum(b + n for b, n in seqs)
            read += mix + used * expert + r["experts"] * h
            flops += 2.0 * (mix + r["top"] * expert + r["experts"] * h) * tokens
    return {"bytes": size * (read + vocab * h + cache + tokens * h) + 4.0 * wanted * vocab,
            "flops": flops + 2.0 * vocab * h * wanted}


def tolerance(case):
    if case["kind"] == "sampling":
        return "exact"
    if case["model"].endswith("float32"):
        return {"rel": 1.5e-5, "max": 2e-4}      # (4e-6 off the 64-bit result)
    if case["model"] == "sosuvik-4k":     # (four layers: 0.004 off the 64-bit result)
        return {"rel": 0.015, "max": 0.15}
    return {"rel": 0.03, "max": 0.3}      # (36 layers of bfloat16 activations: 0.009 to 0.014 off)


# ---------------------------------------------------------------------------------------------------- the same in 64 bits
def _norm(x, w, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _turn(x, rot, adjacent):
    """The first ``dims`` channels of every head of x [T, heads, d] turned by position * frequency."""
    n, base, s = rot["dims"], rot["base"], rot.get("scaling")
    i = torch.arange(n // 2, dtype=F64, device=x.device)
    freq, size = base ** (-2.0 * i / n), 1.0
    if s:
        place = lambda turns: n * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
        low, high = max(math.floor(place(s["fast"])), 0), min(math.ceil(place(s["slow"])), n - 1)
        ramp = ((i - low) / max(high - low, 0.001)).clamp(0.0, 1.0)
        freq, size = freq / s["factor"] * ramp + freq * (1.0 - ramp), 0.1 * math.log(s["factor"]) + 1.0
    angle = torch.arange(x.shape[0], dtype=F64, device=x.device).view(-1, 1, 1) * freq
    cos, sin = angle.cos() * size, angle.sin() * size
    a, b = (slice(0, n, 2), slice(1, n, 2)) if adjacent else (slice(0, n // 2), slice(n // 2, n))
    out = x.clone()
    out[..., a], out[..., b] = x[..., a] * cos - x[..., b] * sin, x[..., b] * cos + x[..., a] * sin
    return out


def _attend(q, k, v, scale, chunk=0, cap=0.0, extra=False):
    """Softmax attention of q [T, heads, d] to k [T, groups, d], v [T, groups, dv]: earlier keys (of the same chunk)."""
    t, heads, groups = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty((t, heads, v.shape[2]), dtype=F64, device=q.device)
    per = heads // groups
    for g in range(groups):
        for r0 in range(0, t, 2048):
            r1 = min(t, r0 + 2048)
            lo = r0 // chunk * chunk if chunk else 0
            s = torch.matmul(q[r0:r1, g * per:(g + 1) * per].transpose(0, 1).contiguous(), k[lo:r1, g].T.contiguous()) * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            i, j = torch.arange(r0, r1, device=q.device).view(-1, 1), torch.arange(lo, r1, device=q.device).view(1, -1)
            seen = (j <= i) & (i // chunk == j // chunk) if chunk else j <= i
            s = s.masked_fill(~seen, float("-inf"))
            top = s.amax(-1, keepdim=True)
            top = top.clamp(min=0.0) if extra else top
            e = torch.exp(s - top)
            den = e.sum(-1, keepdim=True) + (torch.exp(-top) if extra else 0.0)
            out[r0:r1, g * per:(g + 1) * per] = torch.matmul(e / den, v[lo:r1, g].contiguous()).transpose(0, 1)
    return out


def _qwen(get, c, bounds, x):
    d, nq, nkv = QWEN_REST["head_dim"], c["num_attention_heads"], c["num_key_value_heads"]
    rot = {"dims": d, "base": QWEN_REST["rope_theta"]}
    for layer in range(c["num_hidden_layers"]):
        w = lambda name: get(f"model.layers.{layer}.{name}.weight")
        n = _norm(x, w("input_layernorm"))
        q = _norm((n @ w("self_attn.q_proj").T).view(-1, nq, d), w("self_attn.q_norm"))
        k = _norm((n @ w("self_attn.k_proj").T).view(-1, nkv, d), w("self_attn.k_norm"))
        v = (n @ w("self_attn.v_proj").T).view(-1, nkv, d)
        o = torch.cat([_attend(_turn(q[a:b], rot, True), _turn(k[a:b], rot, True), v[a:b], d ** -0.5) for a, b in bounds])
        x = x + o.flatten(1) @ w("self_attn.o_proj").T
        n = _norm(x, w("post_attention_layernorm"))
        g = n @ w("mlp.gate_proj").T
        g = g / (1.0 + torch.exp(-g))
        g *= n @ w("mlp.up_proj").T
        x = x + g @ w("mlp.down_proj").T
    return x


def _experts(n, get, p, e):
    r, limit = e["router"], e["expert"]["limit"]
    score = torch.sigmoid(n @ get(p + "router").T)
    by = score + get(p + "correction")
    count, keep = r["groups"]["count"], r["groups"]["keep"]
    marks = by.view(len(by), count, -1).sort(dim=-1, descending=True).values[..., :2].sum(-1)
    best = marks.sort(dim=-1, descending=True, stable=True).indices[:, :keep]
    allowed = torch.zeros_like(marks, dtype=torch.bool).scatter_(1, best, True).repeat_interleave(r["experts"] // count, 1)
    chosen = by.masked_fill(~allowed, float("-inf")).sort(dim=-1, descending=True, stable=True).indices[:, :r["top"]]
    weight = score.gather(1, chosen)
    weight = weight / (weight.sum(-1, keepdim=True) + 1e-20) * r["scale"]
    out = torch.zeros_like(n)
    for j in range(r["experts"]):
        token, place = (chosen == j).nonzero(as_tuple=True)
        if token.numel():
            h = n[token]
            g = (h @ get(f"{p}e{j}.gate").T).clamp(max=limit)
            u = (h @ get(f"{p}e{j}.up").T).clamp(-limit, limit)
            out[token] += weight[token, place].view(-1, 1) * ((g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ get(f"{p}e{j}.down").T)
    return out


def _sosuvik(get, c, bounds, x):
    first, loop = x, c["loop"]
    order = list(range(loop["start"])) + list(range(loop["start"], loop["stop"])) * loop["times"] + \
        list(range(loop["stop"], len(c["layers"])))
    passes = 0
    for layer in order:
        if layer == loop["start"]:
            x = torch.cat([x, first], -1) @ get("loop.in").T + get("loop.step")[passes]
            passes += 1
        spec, p = c["layers"][layer], f"l{layer}."
        m, t = spec["mixer"], x.shape[0]
        n = _norm(x, get(p + "norm1"))
        if spec["type"] == "attention":
            q, k, v = ((n @ get(p + "mix." + a).T).view(t, h, -1) for a, h in (("q", m["heads"]), ("k", m["kv_heads"]), ("v", m["kv_heads"])))
            o = torch.cat([_attend(_turn(q[a:b], m["rot"], False), _turn(k[a:b], m["rot"], False), v[a:b], m["scale"],
                                   m["mask"]["size"], m["softcap"], True) for a, b in bounds])
        else:
            d, heads, rank = m["dim"], m["heads"], m["kv_rank"]
            q, down = (n @ get(p + "mix.q").T).view(t, heads, -1), n @ get(p + "mix.dkv").T
            row = _norm(down[:, :rank], get(p + "mix.dkv.norm"))
            k, v = ((row @ get(p + "mix." + a).T).view(t, heads, -1) for a in ("uk", "uv"))
            kt = down[:, rank:].unsqueeze(1)
            o = torch.cat([_attend(torch.cat([q[a:b, :, :d], _turn(q[a:b, :, d:], m["rot"], True)], -1),
                                   torch.cat([k[a:b], _turn(kt[a:b], m["rot"], True).expand(-1, heads, -1)], -1), v[a:b], m["scale"])
                           for a, b in bounds])
        x = x + o.flatten(1) @ get(p + "mix.o").T + _experts(_norm(x, get(p + "norm2")), get, p + "mlp.", spec["mlp"])
    return x


def exact(case, seed):
    if case["kind"] == "sampling":
        return None       # whole numbers: the tokens
    source = Checkpoint(case["model"], seed)
    get = lambda name: source.get(name).to(F64)
    contexts, steps, prompts = _traffic(case, seed)
    seqs = [c + [t] for c, t in zip(contexts, steps[0])] + prompts
    ends = np.cumsum([len(s) for s in seqs]).tolist()
    bounds = list(zip([0] + ends[:-1], ends))
    ids = torch.tensor([t for s in seqs for t in s], device=DEVICE)
    last = torch.tensor(ends, device=DEVICE) - 1
    if case["model"] in QWEN:
        x = _qwen(get, QWEN[case["model"]], bounds, source.get("model.embed_tokens.weight")[ids].to(F64))
        return _norm(x[last], get("model.norm.weight")) @ get("lm_head.weight").T
    x = _sosuvik(get, SOSUVIK, bounds, source.get("embed")[ids].to(F64))
    return _norm(x[last], get("final.norm")) @ get("head").T * SOSUVIK["logit_scale"]
