"""The work that users of this engine have it do, as cases whose time and results can be measured.

One pass is a short piece of serving through the step function, driven by :class:`dli_amd.trace.TraceSession` (the
session behind ``bin/trace_run``): requests go on from contexts that lie in the cache, or bring new prompts, or both in
one step; then every request decodes some tokens, one step each, through the recorded decode graphs. The tokens are
given, so that every pass computes the same logits; these are the outputs, one ``[requests, vocabulary]`` tensor a step.

Fields of a case:
  model     sizes, by the names that :data:`LLAMA` and :func:`_config` know; ``dtype``: "bfloat16" or "float32"
  live      requests that go on from a cached context of (up to) ``context`` tokens, with ``bring`` tokens each
  prompts   requests that bring a new prompt of (up to) ``prompt`` tokens in the same step
  steps     decode steps of all requests after that one
  ragged    lengths spread between a quarter and all of ``context`` and ``prompt``, else all of them that long
"""

from __future__ import annotations

import math
import random
import zlib

import torch

from dli_amd.engine.core import build_core
from dli_amd.parts.base import Runtime
from dli_amd.trace import TraceSession
from dli_amd.weights.loader import build_model

PAGE = 16
F = torch.float64

# ------------------------------------------------------------------------------ models

_LLAMA3_ROPE = {"rope_type": "llama3", "factor": 32.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                "original_max_position_embeddings": 8192}
#: name: (vocabulary, width, feed-forward, layers, heads, kv heads, head size, rotary base, scaling)
LLAMA = {
    "SmolLM2-135M": (49152, 576, 1536, 30, 9, 3, 64, 100000.0, None),
    "SmolLM2-360M": (49152, 960, 2560, 32, 15, 5, 64, 100000.0, None),
    "SmolLM2-1.7B": (49152, 2048, 8192, 24, 32, 32, 64, 130000.0, None),
    "Llama-3.2-1B": (128256, 2048, 8192, 16, 32, 8, 64, 500000.0, _LLAMA3_ROPE),
    "Llama-3.2-3B": (128256, 3072, 8192, 28, 24, 8, 128, 500000.0, _LLAMA3_ROPE),
}
#: the other designs' sizes: width, heads (of 64), kv heads, feed-forward, layers, vocabulary, attention chunk
DESIGN_SIZES = {"1024": (1024, 16, 4, 4096, 8, 32000, 1024), "2048": (2048, 32, 8, 8192, 8, 32000, 2048)}


def _config(model):
    """The config.json of a case's model: one of the Llama sizes, or ``Design-width`` with the layers of this
    repository's own benchmark. Feed-forwards are the dense ones, or the experts that a table chooses: a learned router's
    close calls go one way or the other with the last bit of a sum, and then whole rows differ."""
    if model in LLAMA:
        vocab, width, ff, layers, heads, kv, dim, base, scaling = LLAMA[model]
        return {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "vocab_size": vocab, "hidden_size": width,
                "intermediate_size": ff, "num_hidden_layers": layers, "num_attention_heads": heads,
                "num_key_value_heads": kv, "head_dim": dim, "rms_norm_eps": 1e-5, "max_position_embeddings": 131072,
                "rope_theta": base, **({"rope_scaling": scaling} if scaling else {}), "tie_word_embeddings": True,
                "hidden_act": "silu"}
    design, size = model.split("-")
    width, heads, kv, ff, layers, vocab, chunk = DESIGN_SIZES[size]
    if design == "Makodra":
        def layer(kind):
            mixer = {"heads": heads, "dim": 64, "rank": 64} if kind != "attention" else {
                "heads": heads, "kv_heads": kv, "dim": 64, "vdim": 64, "scale": 0.125, "v_mix": True, "mask": {"size": chunk}}
            return {"type": kind, "mixer": mixer, "mlp": {"kind": "dense", "ff": ff}}
        kinds = ("attention", "general_delta", "general_delta", "wkv")
        more = {"logit_softcap": 30.0}
    elif design == "Miberax":
        def layer(kind):
            left = {"heads": heads, "kv_heads": kv, "dim": 64, "vdim": 64, "scale": 0.125, "mask": {"size": chunk},
                    "rot": {"dims": 64, "base": 1e6, "scaling": {"factor": 2.0}}}
            right = {"heads": heads, "kv_heads": kv, "dim": 64, "vdim": 64, "conv": 4}
            return {"type": kind, "mixer": {"left": left, "right": right}, "mlp": {"kind": "dense", "ff": ff}}
        kinds, more = ("parallel",), {}
    elif design == "Rurorax":
        def layer(kind):
            mixer = {"heads": 2 * width // 64, "vdim": 64, "state": 128, "groups": kv, "norm_groups": kv, "conv": 4}
            if kind == "attention":
                mixer = {"heads": heads, "kv_heads": kv, "dim": 64, "vdim": 64, "scale": 0.125, "mask": {"size": chunk},
                         "rot": {"dims": 32, "base": 1e6, "scaling": {"factor": 2.0}}}
            return {"type": kind, "mixer": mixer, "mlp": {"kind": "dense", "ff": ff}}
        kinds, more = ("mamba2", "attention"), {"logit_softcap": 30.0}
    else:
        rot = {"dims": 32, "base": 5e5, "scaling": {"factor": 4.0, "low": 1.0, "high": 4.0, "original": 8192}}
        diff = {"heads": heads // 2, "kv_heads": max(1, kv // 2), "dim": 64, "vdim": 128, "scale": 0.125, "diff": 0.4,
                "mask": {"size": chunk, "keep_first": 64}, "rot": rot}
        pair = {"left": {"heads": heads, "kv_heads": kv, "dim": 64, "vdim": 64, "scale": 0.125, "mask": {"size": chunk},
                         "rot": {"dims": 64, "base": 1e6}},
                "right": {"heads": heads, "dim": 64, "vdim": 64, "decay": [1.0 - 2.0 ** -(3 + 5 * h / heads) for h in range(heads)]},
                "left_scale": 0.7, "right_scale": 0.6}
        mixers = {"attention": diff, "parallel": pair, "mlstm": {"heads": heads, "dim": 64, "vdim": 64, "gate_cap": 10.0}}
        mlp = {"kind": "moe", "expert": {"ff": ff // 8}, "router": {"experts": 32, "top": 4}, "shared": {"ff": ff // 4}}
        kinds, more = ("attention", "parallel", "mlstm", "attention"), {"logit_scale": 0.5}
        chain = [{"type": kinds[i % 4], "mixer": dict(diff, kv_from=i - 3) if i % 4 == 3 else mixers[kinds[i % 4]], "mlp": mlp}
                 for i in range(layers)]
        return {"architecture": design, "vocab": vocab, "width": width, "norm": {"eps": 1e-6}, **more, "layers": chain}
    return {"architecture": design, "vocab": vocab, "width": width,
            "norm": {"eps": 1e-6, **({"groups": 4} if design == "Miberax" else {})}, **more,
            "layers": [layer(kinds[i % len(kinds)]) for i in range(layers)]}


def _shapes(cfg):
    """Name -> shape of every tensor of the checkpoint."""
    if "layers" not in cfg:
        w, ff = cfg["hidden_size"], cfg["intermediate_size"]
        q, kv = (cfg[n] * cfg["head_dim"] for n in ("num_attention_heads", "num_key_value_heads"))
        out = {"model.embed_tokens.weight": (cfg["vocab_size"], w), "model.norm.weight": (w,)}
        for i in range(cfg["num_hidden_layers"]):
            sizes = {"input_layernorm": (w,), "post_attention_layernorm": (w,), "self_attn.q_proj": (q, w),
                     "self_attn.k_proj": (kv, w), "self_attn.v_proj": (kv, w), "self_attn.o_proj": (w, q),
                     "mlp.gate_proj": (ff, w), "mlp.up_proj": (ff, w), "mlp.down_proj": (w, ff)}
            out.update({f"model.layers.{i}.{n}.weight": s for n, s in sizes.items()})
        return out
    w, design = cfg["width"], cfg["architecture"]
    out = {"embed": (cfg["vocab"], w), "final.norm": (w,)}
    if design == "Rurorax":
        out.update({"final.norm.b": (w,), "final.norm.alpha": ()})
    if design == "Betepel":
        out["embed.norm"] = (w,)

    def attention(p, m, maps=1, bias=False, own=True):
        H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        sizes = {"q": H * maps * D, **({"k": G * maps * D, "v": G * V} if own else {})}
        out.update({p + n: (rows, w) for n, rows in sizes.items()})
        if bias:
            out.update({p + n + ".b": (rows,) for n, rows in sizes.items()})
        out[p + "o"] = (w, H * V)

    for i, layer in enumerate(cfg["layers"]):
        p, m, kind, f = f"l{i}.mix.", layer["mixer"], layer["type"], layer["mlp"]
        out.update({f"l{i}.norm1": (w,)})
        if design != "Rurorax":
            out[f"l{i}.norm2"] = (w,)
        if design == "Makodra":
            H, c = m["heads"], m["heads"] * m["dim"]
            if kind == "attention":
                attention(p, m)
                out.update({p + "g": (H * m["vdim"], w), p + "r1": (H,), p + "r2": (H,), p + "vmix": ()})
            else:
                out.update({p + s: (c, w) for s in "rkvg"})
                out.update({p + "w1": (m["rank"], w), p + "w2": (c, m["rank"]), p + "w0": (c,), p + "norm": (c,), p + "o": (w, c)})
                out.update({p + "a": (c, w), p + "a.b": (c,)} if kind == "general_delta" else
                           {**{p + "mu." + s: (w,) for s in "rkvgw"}, p + "u": (H, m["dim"])})
        elif design == "Miberax":
            attention(p + "left.", m["left"])
            d, r = m["right"], p + "right."
            qk, hv = d["kv_heads"] * d["dim"], d["heads"] * d["vdim"]
            out.update({p + "left.out": (w,), r + "out": (w,), r + "q": (qk, w), r + "k": (qk, w), r + "v": (hv, w),
                        r + "q.conv": (qk, d["conv"]), r + "k.conv": (qk, d["conv"]), r + "v.conv": (hv, d["conv"]),
                        r + "b": (d["heads"], w), r + "a": (d["heads"], w), r + "A_log": (d["heads"],),
                        r + "dt_bias": (d["heads"],), r + "norm": (d["vdim"],), r + "g": (hv, w), r + "o": (w, hv)})
        elif design == "Rurorax":
            out.update({f"l{i}.norm1.b": (w,), f"l{i}.norm1.alpha": (), f"l{i}.ls1": (w,), f"l{i}.ls2": (w,)})
            if kind == "attention":
                attention(p, m, bias=True)
                out.update({p + "q.norm": (m["heads"] * m["dim"],), p + "k.norm": (m["kv_heads"] * m["dim"],), p + "o.b": (w,)})
            else:
                H, inner = m["heads"], m["heads"] * m["vdim"]
                channels = inner + 2 * m["groups"] * m["state"]
                out.update({p + "in": (inner + channels + H, w), p + "conv": (channels, m["conv"]), p + "conv.b": (channels,),
                            p + "dt_bias": (H,), p + "A_log": (H,), p + "D": (H,), p + "norm": (inner,), p + "o": (w, inner)})
        elif kind == "mlstm":
            H, c = m["heads"], m["heads"] * m["dim"]
            out.update({p + s: (c, w) for s in "qkvg"})
            out.update({p + "o": (w, c), p + "norm": (c,), p + "i": (H, w), p + "f": (H, w), p + "i.b": (H,), p + "f.b": (H,)})
        elif kind == "attention":
            attention(p, m, maps=2, bias=True, own=m.get("kv_from") is None)
            out.update({p + n: (m["dim"],) for n in ("lq1", "lk1", "lq2", "lk2")})
            out[p + "g"] = (m["heads"], w)
        else:
            attention(p + "left.", m["left"], bias=True)
            c = m["right"]["heads"] * m["right"]["dim"]
            out.update({p + "right." + s: (c, w) for s in "qkvg"})
            out.update({p + "right.o": (w, c), p + "right.norm": (c,)})
        q = f"l{i}.mlp."
        if f["kind"] == "moe":
            out[q + "table"] = (cfg["vocab"], f["router"]["top"])
            for e, ff in [(f"e{e}", f["expert"]["ff"]) for e in range(f["router"]["experts"])] + [("shared", f["shared"]["ff"])]:
                out.update({f"{q}{e}.gate": (ff, w), f"{q}{e}.up": (ff, w), f"{q}{e}.down": (w, ff)})
        else:
            out.update({q + "up": (f["ff"], w), q + "down": (w, f["ff"])})
            if design == "Miberax":
                out[q + "act"] = (4,)
            else:
                out[q + "gate"] = (f["ff"], w)
            if design == "Rurorax":
                out.update({q + "gate.b": (f["ff"],), q + "up.b": (f["ff"],), q + "down.b": (w,)})
    return out


def _weights(cfg, seed, device):
    """Every tensor drawn from the seed, with values that bfloat16 holds: matrices with outputs of about the size of
    their inputs, norm weights near one (or near zero where they are offsets), decays and rates spread out. What is
    added to the residual stream is smaller by the root of the number of sums, as in trained models: the stream then
    neither grows from layer to layer nor multiplies its roundings."""
    design, out = cfg.get("architecture"), {}
    sums = 2 * (cfg.get("num_hidden_layers") or len(cfg["layers"]))
    for name, shape in _shapes(cfg).items():
        gen = torch.Generator(device=device).manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (1 << 62))
        leaf = name.split(".")[-1]
        if leaf == "table":
            experts = cfg["layers"][0]["mlp"]["router"]["experts"]
            keys = torch.rand((shape[0], experts), generator=gen, device=device)
            out[name] = keys.argsort(dim=1)[:, :shape[1]].to(torch.int32)
            continue
        r = torch.randn(shape, generator=gen, device=device)
        if leaf in ("norm1", "norm2") or name in ("embed.norm", "final.norm"):
            t = 0.1 * r + (0.0 if design == "Betepel" else 1.0)
            if design == "Makodra" and leaf in ("norm1", "norm2"):   # these scale what is added
                t = t / math.sqrt(sums)
        elif leaf in ("norm", "out") or name.endswith("norm.weight"):
            t = 1.0 + 0.1 * r
            if leaf == "out":
                t = t / math.sqrt(sums)
        elif leaf in ("w0", "A_log", "dt_bias"):
            t = r - {"w0": 0.0, "A_log": 1.0, "dt_bias": 2.0}[leaf]
        elif leaf in ("alpha", "vmix", "r1", "r2", "ls1", "ls2", "D"):
            t = 0.5 + 0.1 * r
        elif name.split(".")[-2:-1] == ["mu"]:
            t = 0.5 + 0.2 * r
        elif leaf == "act":
            t = torch.tensor([1.0, 0.5, -0.3, 0.1], device=device) + 0.1 * r
        elif leaf in ("u", "conv"):
            t = 0.5 * r
        elif name.endswith(("f.b", "i.b")):
            t = r + (2.0 if name.endswith("f.b") else 0.0)
        elif leaf in ("b", "lq1", "lk1", "lq2", "lk2"):
            t = 0.3 * r
        elif "embed" in name or "layers" not in cfg:
            t = (1.0 if "embed" in name else 0.02) * r
        else:
            t = r / math.sqrt(shape[-1])
        if leaf in ("o", "down") and design not in ("Makodra", "Rurorax") or "o_proj" in name or "down_proj" in name:
            t = t / math.sqrt(sums)
        out[name] = t.to(torch.bfloat16)
    return out


# ------------------------------------------------------------------------------ cases

def _case(name, model, *, dtype="bfloat16", live=0, context=0, bring=1, prompts=0, prompt=0, steps=0, ragged=False):
    out = {"name": name, "model": model, "dtype": dtype, "live": live, "context": context, "bring": bring,
           "prompts": prompts, "prompt": prompt, "steps": steps, "ragged": ragged}
    if name is None:
        del out["name"]
    return out


def listed():
    return [
        # a small model answering one user on the device: short kernels, launches and gaps between them
        _case("decode-135m-b1", "SmolLM2-135M", live=1, context=512, steps=7),
        # interactive use of the 1B model: one user, and the batch of eight that the headline number is quoted on
        _case("decode-1b-b1", "Llama-3.2-1B", live=1, context=4096, steps=7),
        _case("decode-1b-b8", "Llama-3.2-1B", live=8, context=4096, steps=7),
        # a loaded server: 64 requests that are at different places of their conversations
        _case("decode-1b-b64-ragged", "Llama-3.2-1B", live=64, context=4096, steps=7, ragged=True),
        # time to the first token of a usual prompt, and of a long one on the largest sizes
        _case("prompt-1b-2048", "Llama-3.2-1B", prompts=1, prompt=2048),
        _case("prompt-3b-8192", "Llama-3.2-3B", prompts=1, prompt=8192),
        # continuous batching: portions of prompts beside single tokens in one step (as many kv heads as heads)
        _case("mixed-1.7b", "SmolLM2-1.7B", live=24, context=1024, prompts=3, prompt=611, steps=2, ragged=True),
        # the 32-bit path, which results are compared on
        _case("fp32-135m", "SmolLM2-135M", dtype="float32", prompts=2, prompt=333, steps=4, ragged=True),
        # the other designs: a prompt or a few of them, then the reply's first tokens
        _case("makodra-prompt-2048", "Makodra-2048", prompts=1, prompt=2048, steps=4),
        _case("miberax-4-prompts", "Miberax-2048", prompts=4, prompt=1100, steps=8, ragged=True),
        _case("betepel-2-prompts", "Betepel-2048", prompts=2, prompt=1500, steps=8, ragged=True),
        _case("rurorax-prompt-4096", "Rurorax-2048", prompts=1, prompt=4096, steps=4),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng: random.Random):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "mixed", "fp32", "design", "design"])
    llama = rng.choice(sorted(LLAMA))
    if kind == "decode":
        live = _log(rng, 1, 64)
        context = min(_log(rng, 48, 8192), 262144 // live // (2 if "B" in llama and llama != "Llama-3.2-1B" else 1))
        return _case(None, llama, live=live, context=context, steps=rng.randint(3, 8), ragged=rng.random() < 0.5)
    if kind == "prompt":
        prompts = _log(rng, 1, 8)
        return _case(None, llama, prompts=prompts, prompt=_log(rng, 17, 8192 // prompts), steps=rng.choice([0, 0, 1, 4]),
                     ragged=rng.random() < 0.5)
    if kind == "mixed":
        return _case(None, llama, live=_log(rng, 1, 40), context=_log(rng, 64, 2048), bring=rng.choice([1, 1, rng.randint(2, 60)]),
                     prompts=rng.randint(1, 4), prompt=_log(rng, 17, 1500), steps=rng.randint(0, 4), ragged=True)
    if kind == "fp32":
        return _case(None, rng.choice(["SmolLM2-135M", "SmolLM2-360M"]), dtype="float32", prompts=rng.randint(1, 4),
                     prompt=_log(rng, 17, 500), steps=rng.randint(0, 4), ragged=True)
    design, size = rng.choice(["Makodra", "Miberax", "Betepel", "Rurorax"]), rng.choice(sorted(DESIGN_SIZES))
    prompts = _log(rng, 1, 16)
    return _case(None, f"{design}-{size}", prompts=prompts, prompt=_log(rng, 33, 6000 // prompts), steps=rng.randint(0, 8),
                 ragged=rng.random() < 0.5)


def _lengths(count, most, ragged, multiple=1):
    """Lengths of ``count`` contexts or prompts, whole multiples of ``multiple`` (at least one)."""
    out = []
    for i in range(count):
        n = most * (1.0 - 0.75 * ((i * 0.6180339887) % 1.0)) if ragged else most
        out.append(max(1, int(n) // multiple) * multiple)
    return out


def _requests(case):
    """Per request: tokens in the cache before the pass, and tokens that it brings in the pass's first step. Contexts
    end at a page's end: what continues them starts a page of its own."""
    live = [(n, case["bring"]) for n in _lengths(case["live"], case["context"], case["ragged"], PAGE)]
    return live + [(0, n) for n in _lengths(case["prompts"], case["prompt"], case["ragged"])]


def _tokens(case, vocab, seed):
    """Per request, all its tokens: context, then those of the pass."""
    gen = torch.Generator().manual_seed(seed)
    return [torch.randint(0, vocab, (old + new + case["steps"],), generator=gen).tolist() for old, new in _requests(case)]


def prepare(case, seed):
    """A loaded model, its engine core, the contexts in its cache, and one pass as a server's warm-up (which records
    the decode graphs)."""
    cfg, device = _config(case["model"]), torch.device("cuda")
    dtype = getattr(torch, case["dtype"])
    model, _ = build_model(cfg, Runtime(device, dtype))
    drawn = _weights(cfg, seed, device)
    kinds = {"matrix": dtype, "float32": torch.float32, "int32": torch.int32}
    model.load_weights({n: drawn[n].to(kinds[s.role]) for n, s in model.weight_specs().items() if n in drawn})
    requests = _requests(case)
    tokens = _tokens(case, cfg.get("vocab_size") or cfg["vocab"], seed)
    longest = max(old + new for old, new in requests) + case["steps"]
    pages = sum(-(-old // PAGE) + -(-(new + case["steps"]) // PAGE) for old, new in requests) + len(requests) + 8
    core = build_core(model, num_pages=pages, page_size=PAGE, max_seqs=len(requests) + case["live"],
                      enable_prefix_caching=False, watermark=0.0)
    core.step.enable_decode_graphs(len(requests), longest)
    session = TraceSession(core)
    batch = []
    for i in range(case["live"]):
        batch.append({"id": f"context {i}", "tokens": tokens[i][:requests[i][0]]})
        if i + 1 == case["live"] or sum(len(e["tokens"]) for e in batch) + requests[i + 1][0] > 16384:
            session.step(batch)
            batch = []
    entries, decodes = [], []
    for i, (old, new) in enumerate(requests):
        entries.append({"id": f"r{i}", "tokens": tokens[i][old:old + new], "want": [new - 1]})
    for j in range(case["steps"]):
        decodes.append([{"id": f"r{i}", "tokens": [tokens[i][old + new + j]], "want": [0]} for i, (old, new) in enumerate(requests)])
    state = {"session": session, "live": case["live"], "rounds": [entries] + decodes}
    run(state)
    return state


def run(state):
    """One pass: the contexts' continuations begin, all requests run their steps and end. (Logits of a replayed step lie
    in the graph's own buffer until the next one: whoever keeps them copies them.)"""
    session, rounds, out = state["session"], state["rounds"], []
    for i in range(state["live"]):
        session.fork(f"context {i}", f"r{i}")
    for j, entries in enumerate(rounds):
        last = j + 1 == len(rounds)
        out.append(session.step(entries, [e["id"] for e in entries] if last else ()).clone())
    return out


def work(case):
    """Bytes: every weight once a step (the rows of the embedding that are read aside), the keys and values that the
    step's queries see, the logits. Operations: two a weight and token, and the attention's products. Steps follow one
    another, so a step's weights cannot be kept for the next."""
    cfg, requests = _config(case["model"]), _requests(case)
    item = 2 if case["dtype"] == "bfloat16" else 4
    sizes = {n: math.prod(s) for n, s in _shapes(cfg).items()}
    experts = sum(v for n, v in sizes.items() if ".mlp.e" in n)
    table = sum(v for n, v in sizes.items() if n.endswith("table"))
    head = sizes.get("model.embed_tokens.weight", 0) or sizes["embed"]
    dense = sum(sizes.values()) - experts - table - head
    vocab = cfg.get("vocab_size") or cfg["vocab"]
    # per attention layer: (values of keys and values a token, multiplications a query and key, how far it sees)
    layers = []
    if "layers" not in cfg:
        h, g, d = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
        layers = [(2 * g * d, 2 * h * d, 0)] * cfg["num_hidden_layers"]
    else:
        for layer in cfg["layers"]:
            m = layer["mixer"].get("left", layer["mixer"])
            if "kv_heads" in m:
                maps = 2 if "diff" in m else 1
                layers.append((m["kv_heads"] * (maps * m["dim"] + m["vdim"]), maps * m["heads"] * (m["dim"] + m["vdim"]), m["mask"]["size"]))
    total, flops = 0.0, 0.0
    for step in range(1 + case["steps"]):
        rows = [(old + (0 if step == 0 else new + step - 1), new if step == 0 else 1) for old, new in requests]
        n = sum(new for _, new in rows)
        top = 4 * n
        used = experts * min(1.0, 1.0 - (1.0 - 1.0 / 32) ** top) if experts else 0.0
        total += (dense + head + used) * item + len(rows) * vocab * 4
        flops += 2.0 * n * (dense + experts / 32 * 4) + 2.0 * len(rows) * head
        for kv, products, size in layers:
            for old, new in rows:
                # keys that a portion's queries see between them, and pairs of query and key
                seen = min(old + new, new + size - 1) if size else old + new
                pairs = new * old + new * (new + 1) / 2
                total += seen * kv * item
                flops += 2.0 * products * (min(pairs, float(new) * size) if size else pairs)
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Logits after many layers in bfloat16, with 32-bit sums, lie 0.3e-2 (Betepel) to 1.2e-2 from exact ones, and two
    right implementations as far from each other. In 32-bit 0.4e-6 with sums in runs of 256 terms; in one run the
    rounding of sums of up to 1,536 terms through 30 layers is about three times that."""
    return {"rel": 4e-6, "max": 2e-4} if case["dtype"] == "float32" else {"rel": 0.025}


# ------------------------------------------------------------------------------ the same in 64 bits, by plain torch

def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _attend(q, k, v, scale, *, chunk=0, window=0, keep=0, sink=False, penalty=None):
    """Causal attention of one sequence: ``q [n, H, D]``, ``k [n, G, D]``, ``v [n, G, V]`` -> ``[n, H, V]``. ``chunk``: only
    keys of the query's chunk; ``window``: only that many keys up to the query, and the first ``keep``; ``sink``: one is
    added to the sum of exponentials; ``penalty``: ``r1 log(1 + r2 distance)`` off the scores."""
    n, H, _ = q.shape
    G = k.shape[1]
    out = torch.empty(n, H, v.shape[2], dtype=F, device=q.device)
    kt, vg, pos = k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous(), torch.arange(n, device=q.device)
    for a in range(0, n, 256):
        b = min(n, a + 256)
        lo = a // chunk * chunk if chunk else 0
        i, j = pos[a:b, None], pos[None, lo:b]
        ok = j <= i
        if chunk:
            ok = ok & (i // chunk == j // chunk)
        if window:
            ok = ok & ((i - j < window) | (j < keep))
        s = q[a:b].view(b - a, G, H // G, -1).permute(1, 2, 0, 3).reshape(G, -1, q.shape[2]) @ kt[:, :, lo:b] * scale
        s = s.view(H, b - a, b - lo)
        if penalty is not None:
            s = s - penalty[0][:, None, None] * torch.log1p(penalty[1][:, None, None] * (i - j).clamp(min=0).to(F))
        s = s.masked_fill(~ok, -math.inf)
        e = torch.exp(s) if sink else torch.exp(s - s.amax(-1, keepdim=True))
        e = e / (e.sum(-1, keepdim=True) + (1.0 if sink else 0.0))
        o = e.view(G, -1, b - lo) @ vg[:, lo:b]
        out[a:b] = o.view(G, H // G, b - a, -1).permute(2, 0, 1, 3).reshape(b - a, H, -1)
    return out


def _llama_frequencies(cfg, device):
    """The rotary frequencies, in the 32-bit arithmetic that the architecture fixes for them."""
    d = cfg["head_dim"]
    f = 1.0 / (cfg["rope_theta"] ** (torch.arange(0, d, 2, dtype=torch.int64).to(torch.float32) / d))
    s = cfg.get("rope_scaling")
    if s:
        old, wave = s["original_max_position_embeddings"], 2 * math.pi / f
        low, high = old / s["low_freq_factor"], old / s["high_freq_factor"]
        t = (old / wave - s["low_freq_factor"]) / (s["high_freq_factor"] - s["low_freq_factor"])
        f = torch.where(wave < high, f, torch.where(wave > low, f / s["factor"], (1 - t) * f / s["factor"] + t * f))
    return f.to(device)


def _rotate(x, freq, interleaved=False, angle_type=F):
    """The first components of every head turned by their position's angles: ``i`` with ``i + half``, or in neighbours."""
    n, half = x.shape[0], freq.shape[0]
    angle = (torch.arange(n, device=x.device).to(angle_type)[:, None] * freq.to(angle_type)).to(F)[:, None]
    c, s = torch.cos(angle), torch.sin(angle)
    if interleaved:
        a, b = x[..., 0:2 * half:2], x[..., 1:2 * half:2]
        return torch.cat([torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2), x[..., 2 * half:]], -1)
    a, b = x[..., :half], x[..., half:2 * half]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., 2 * half:]], -1)


def _frequencies(rot, device):
    i = torch.arange(rot["dims"] // 2, dtype=F)
    f, s = torch.pow(torch.tensor(rot["base"], dtype=F), -2.0 * i / rot["dims"]), rot.get("scaling") or {}
    if "original" in s:
        wave = 2 * math.pi / f
        t = (s["original"] / wave - s["low"]) / (s["high"] - s["low"])
        f = torch.where(wave < s["original"] / s["high"], f,
                        torch.where(wave > s["original"] / s["low"], f / s["factor"], (1 - t) * f / s["factor"] + t * f))
    else:
        f = f / s.get("factor", 1.0)
    return f.to(device)


def _scan(n, shape, device, step):
    """``step(t, S) -> S, o`` for every token, from a state of zeros; the ``o`` one below the other."""
    S, out = torch.zeros(shape, dtype=F, device=device), []
    for t in range(n):
        S, o = step(t, S)
        out.append(o)
    return torch.stack(out)


def _rows(S, x):
    """``S^T x`` a head: ``S [H, D, V]``, ``x [H, D]`` -> ``[H, V]``."""
    return (S * x[:, :, None]).sum(1)


def _conv(x, w):
    """Causal convolution per channel: ``x [n, c]``, ``w [c, taps]``, zeros before the start."""
    n, taps = x.shape[0], w.shape[1]
    full = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
    return sum(full[j:j + n] * w[:, j] for j in range(taps))


def _llama(cfg, T, ids):
    n, eps, d = len(ids), cfg["rms_norm_eps"], cfg["head_dim"]
    H, G = cfg["num_attention_heads"], cfg["num_key_value_heads"]
    freq = _llama_frequencies(cfg, ids.device)
    x = T("model.embed_tokens.weight", rows=ids)
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = _rms(x, eps) * T(p + "input_layernorm.weight")
        q, k, v = (h @ T(f"{p}self_attn.{s}_proj.weight").T for s in "qkv")
        q, k = (_rotate(t.view(n, -1, d), freq, angle_type=torch.float32) for t in (q, k))
        x = x + _attend(q, k, v.view(n, G, d), d ** -0.5).view(n, H * d) @ T(p + "self_attn.o_proj.weight").T
        h = _rms(x, eps) * T(p + "post_attention_layernorm.weight")
        x = x + (_silu(h @ T(p + "mlp.gate_proj.weight").T) * (h @ T(p + "mlp.up_proj.weight").T)) @ T(p + "mlp.down_proj.weight").T
    return lambda rows: (_rms(x[rows], eps) * T("model.norm.weight")) @ T("model.embed_tokens.weight").T


def _makodra(cfg, T, ids):
    n, eps, w, first = len(ids), cfg["norm"]["eps"], cfg["width"], None
    i = torch.arange(w // 2, dtype=F, device=ids.device)
    angle = torch.arange(n, device=ids.device).to(F)[:, None] * torch.pow(torch.tensor(10000.0, dtype=F, device=ids.device), -2.0 * i / w)
    x = T("embed", rows=ids) + torch.stack([torch.sin(angle), torch.cos(angle)], -1).flatten(-2)
    for l, layer in enumerate(cfg["layers"]):
        p, m = f"l{l}.mix.", layer["mixer"]
        H, D = m["heads"], m["dim"]
        if layer["type"] == "attention":
            q, k = (_rms((x @ T(p + s).T).view(n, -1, D), eps) for s in "qk")
            v = (x @ T(p + "v").T).view(n, -1, m["vdim"])
            first, v = (v, v) if first is None else (first, (1 - T(p + "vmix")) * v + T(p + "vmix") * first)
            o = _attend(q, k, v, m["scale"], chunk=m["mask"]["size"], sink=True, penalty=(T(p + "r1"), T(p + "r2")))
            y = (o.reshape(n, -1) * torch.sigmoid(x @ T(p + "g").T)) @ T(p + "o").T
        else:
            delta = layer["type"] == "general_delta"
            before = torch.cat([torch.zeros_like(x[:1]), x[:-1]])
            mix = (lambda s: x) if delta else (lambda s: x + (before - x) * T(p + "mu." + s))
            r, k, v = ((mix(s) @ T(p + s).T).view(n, H, D) for s in "rkv")
            low = torch.tanh(mix("w") @ T(p + "w1").T) @ T(p + "w2").T + T(p + "w0")
            if delta:
                decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(low)).view(n, H, D)
                u = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
                au = torch.sigmoid(x @ T(p + "a").T + T(p + "a.b")).view(n, H, D) * u

                def step(t, S):
                    S = decay[t][:, :, None] * S - au[t][:, :, None] * _rows(S, u[t])[:, None] + k[t][:, :, None] * v[t][:, None]
                    return S, _rows(S, r[t])
            else:
                decay, bonus = torch.exp(-torch.exp(low)).view(n, H, D), T(p + "u")[:, :, None]

                def step(t, S):
                    kv = k[t][:, :, None] * v[t][:, None]
                    return decay[t][:, :, None] * S + kv, _rows(S + bonus * kv, r[t])
            o = _rms(_scan(n, (H, D, D), x.device, step), eps).reshape(n, -1) * T(p + "norm")
            gate = mix("g") @ T(p + "g").T
            y = (o * (torch.sigmoid(gate) if delta else _silu(gate))) @ T(p + "o").T
        x = x + _rms(y, eps) * T(f"l{l}.norm1")
        q = f"l{l}.mlp."
        x = x + _rms((_silu(x @ T(q + "gate").T) * (x @ T(q + "up").T)) @ T(q + "down").T, eps) * T(f"l{l}.norm2")
    cap = cfg["logit_softcap"]
    return lambda rows: cap * torch.tanh((_rms(x[rows], eps) * T("final.norm")) @ T("embed").T / cap)


def _miberax(cfg, T, ids):
    n, eps, groups = len(ids), cfg["norm"]["eps"], cfg["norm"]["groups"]

    def norm(x, name):
        return _rms(x.view(x.shape[0], groups, -1), eps).reshape(x.shape) * T(name)

    def unit(x):
        return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)

    x = T("embed", rows=ids)
    for l, layer in enumerate(cfg["layers"]):
        h, p, a, d = norm(x, f"l{l}.norm1"), f"l{l}.mix.left.", layer["mixer"]["left"], layer["mixer"]["right"]
        freq = _frequencies(a["rot"], ids.device)
        q, k = (_rotate((h @ T(p + s).T).view(n, -1, a["dim"]), freq, interleaved=True) for s in "qk")
        left = _attend(q, k, (h @ T(p + "v").T).view(n, -1, a["vdim"]), a["scale"], chunk=a["mask"]["size"]).reshape(n, -1) @ T(p + "o").T
        left = _rms(left, eps) * T(p + "out")
        p, H, rep = f"l{l}.mix.right.", d["heads"], d["heads"] // d["kv_heads"]
        q, k, v = (_silu(_conv(h @ T(p + s).T, T(f"{p}{s}.conv"))) for s in "qkv")
        q, k = (unit(t.view(n, -1, d["dim"])).repeat_interleave(rep, 1) for t in (q, k))
        q, v = q * d["dim"] ** -0.5, v.view(n, H, -1)
        beta = torch.sigmoid(h @ T(p + "b").T)
        g = torch.exp(-torch.exp(T(p + "A_log")) * torch.nn.functional.softplus(h @ T(p + "a").T + T(p + "dt_bias")))

        def step(t, S):
            S = S * g[t][:, None, None]
            S = S + k[t][:, :, None] * (beta[t][:, None] * (v[t] - _rows(S, k[t])))[:, None]
            return S, _rows(S, q[t])
        o = _rms(_scan(n, (H, d["dim"], d["vdim"]), x.device, step), eps) * T(p + "norm") * _silu((h @ T(p + "g").T).view(n, H, -1))
        x = x + 0.5 * (left + _rms(o.reshape(n, -1) @ T(p + "o").T, eps) * T(p + "out"))
        z = norm(x, f"l{l}.norm2") @ T(f"l{l}.mlp.up").T
        c = T(f"l{l}.mlp.act")
        x = x + (c[0] * _rms(z, eps) + c[1] * _rms(z * z, eps) + c[2] * _rms(z ** 3, eps) + c[3]) @ T(f"l{l}.mlp.down").T
    return lambda rows: norm(x[rows], "final.norm") @ T("embed").T


def _rurorax(cfg, T, ids):
    n, eps = len(ids), cfg["norm"]["eps"]

    def norm(x, name):
        return torch.tanh(T(name + ".alpha") * x) * T(name) + T(name + ".b")

    x = T("embed", rows=ids)
    for l, layer in enumerate(cfg["layers"]):
        p, m, h = f"l{l}.mix.", layer["mixer"], norm(x, f"l{l}.norm1")
        if layer["type"] == "attention":
            freq, D = _frequencies(m["rot"], ids.device), m["dim"]
            q, k = (_rotate((_rms(h @ T(p + s).T + T(f"{p}{s}.b"), eps) * T(f"{p}{s}.norm")).view(n, -1, D), freq) for s in "qk")
            o = _attend(q, k, (h @ T(p + "v").T + T(p + "v.b")).view(n, -1, m["vdim"]), m["scale"], chunk=m["mask"]["size"])
            y = o.reshape(n, -1) @ T(p + "o").T + T(p + "o.b")
        else:
            H, V, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
            z, xbc, dt = (h @ T(p + "in").T).split([H * V, H * V + 2 * G * N, H], 1)
            u, B, C = _silu(_conv(xbc, T(p + "conv")) + T(p + "conv.b")).split([H * V, G * N, G * N], 1)
            u, B, C = u.view(n, H, V), B.reshape(n, G, N), C.reshape(n, G, N)
            dt = torch.nn.functional.softplus(dt + T(p + "dt_bias"))
            decay = torch.exp(-torch.exp(T(p + "A_log")) * dt)
            rep, skip = H // G, T(p + "D")[:, None]

            def step(t, S):
                S = decay[t][:, None, None] * S + (dt[t][:, None] * B[t].repeat_interleave(rep, 0))[:, :, None] * u[t][:, None]
                return S, _rows(S, C[t].repeat_interleave(rep, 0)) + skip * u[t]
            o = _scan(n, (H, N, V), x.device, step).reshape(n, -1) * _silu(z)
            y = (_rms(o.view(n, m["norm_groups"], -1), eps).reshape(n, -1) * T(p + "norm")) @ T(p + "o").T
        q = f"l{l}.mlp."
        gate = h @ T(q + "gate").T + T(q + "gate.b")
        f = torch.nn.functional.gelu(gate, approximate="tanh") * (h @ T(q + "up").T + T(q + "up.b"))
        x = x + T(f"l{l}.ls1") * y + T(f"l{l}.ls2") * (f @ T(q + "down").T + T(q + "down.b"))
    cap = cfg["logit_softcap"]
    return lambda rows: cap * torch.tanh(norm(x[rows], "final.norm") @ T("embed").T / cap)


def _betepel(cfg, T, ids):
    n, eps, kept = len(ids), cfg["norm"]["eps"], {}

    def norm(x, name):
        return _rms(x, eps) * (1.0 + T(name))

    def ffn(h, p):
        return (_silu(h @ T(p + "gate").T) * (h @ T(p + "up").T)) @ T(p + "down").T

    x = norm(T("embed", rows=ids), "embed.norm")
    for l, layer in enumerate(cfg["layers"]):
        p, m, h = f"l{l}.mix.", layer["mixer"], norm(x, f"l{l}.norm1")
        if layer["type"] == "attention":
            freq, D, mask = _frequencies(m["rot"], ids.device), m["dim"], m["mask"]
            q = _rotate((h @ T(p + "q").T + T(p + "q.b")).view(n, -1, D), freq).view(n, -1, 2, D)
            if m.get("kv_from") is None:
                kept[l] = (_rotate((h @ T(p + "k").T + T(p + "k.b")).view(n, -1, D), freq).view(n, -1, 2, D),
                           (h @ T(p + "v").T + T(p + "v.b")).view(n, -1, m["vdim"]))
            k, v = kept[l if m.get("kv_from") is None else m["kv_from"]]
            a = [_attend(q[:, :, s].contiguous(), k[:, :, s], v, m["scale"], window=mask["size"], keep=mask["keep_first"]) for s in (0, 1)]
            lam = [torch.exp((T(f"{p}lq{s}") * T(f"{p}lk{s}")).sum()) for s in (1, 2)]
            o = _rms(a[0] - (lam[0] - lam[1] + m["diff"]) * a[1], eps) * (1.0 - m["diff"])
            y = (o * torch.sigmoid(h @ T(p + "g").T)[:, :, None]).reshape(n, -1) @ T(p + "o").T
        elif layer["type"] == "parallel":
            a, r, s = m["left"], m["right"], p + "left."
            freq, D = _frequencies(a["rot"], ids.device), a["dim"]
            q, k = (_rotate((h @ T(s + t).T + T(f"{s}{t}.b")).view(n, -1, D), freq) for t in "qk")
            left = _attend(q, k, (h @ T(s + "v").T + T(s + "v.b")).view(n, -1, a["vdim"]), a["scale"], window=a["mask"]["size"])
            left, s, H = left.reshape(n, -1) @ T(s + "o").T, p + "right.", r["heads"]
            q, k, v = (_silu(h @ T(s + t).T).view(n, H, -1) for t in "qkv")
            decay = torch.tensor(r["decay"], dtype=F, device=x.device)[:, None, None]

            def step(t, S):
                S = decay * S + k[t][:, :, None] * v[t][:, None]
                return S, _rows(S, q[t])
            o = _rms(_scan(n, (H, r["dim"], r["vdim"]), x.device, step).reshape(n, -1), eps) * T(s + "norm")
            y = m["left_scale"] * left + m["right_scale"] * ((o * torch.sigmoid(h @ T(s + "g").T)) @ T(s + "o").T)
        else:
            H, D, cap = m["heads"], m["dim"], m["gate_cap"]
            q, k, v = ((h @ T(p + s).T).view(n, H, D) for s in "qkv")
            q = q * D ** -0.5
            i, f = (cap * torch.tanh((h @ T(p + s).T + T(f"{p}{s}.b")) / cap) for s in "if")
            f, top = torch.nn.functional.logsigmoid(f), [torch.zeros(H, dtype=F, device=x.device)]

            def step(t, S):  # the last column of S is the normalizer
                new = torch.maximum(f[t] + top[0], i[t])
                keep, write = torch.exp(f[t] + top[0] - new), torch.exp(i[t] - new)
                top[0] = new
                one = torch.cat([v[t], torch.ones_like(v[t][:, :1])], 1)
                S = keep[:, None, None] * S + (write[:, None] * k[t])[:, :, None] * one[:, None]
                o = _rows(S, q[t])
                return S, o[:, :-1] / (torch.maximum(o[:, -1].abs(), torch.exp(-new)) + 1e-6)[:, None]
            o = _rms(_scan(n, (H, D, D + 1), x.device, step), eps).reshape(n, -1) * T(p + "norm")
            y = (o * torch.sigmoid(h @ T(p + "g").T)) @ T(p + "o").T
        e, g, fcfg = norm(x, f"l{l}.norm2"), f"l{l}.mlp.", layer["mlp"]
        top, chosen = fcfg["router"]["top"], T(g + "table", rows=ids).to(torch.long)
        y = y + ffn(e, g + "shared.")
        for j in range(fcfg["router"]["experts"]):
            rows = (chosen == j).any(1).nonzero()[:, 0]
            if len(rows):
                y[rows] += ffn(e[rows], f"{g}e{j}.") / top
        x = x + y
    return lambda rows: (norm(x[rows], "final.norm") @ T("embed").T) * cfg["logit_scale"]


_PLAIN = {"Makodra": _makodra, "Miberax": _miberax, "Rurorax": _rurorax, "Betepel": _betepel}


def exact(case, seed):
    """The pass's logits by whole sequences in float64, on the weights as they are stored."""
    cfg, device = _config(case["model"]), torch.device("cuda")
    stored = _weights(cfg, seed, device)
    plain = _PLAIN.get(cfg.get("architecture"), _llama)
    wide = {}

    def T(name, rows=None):
        if rows is not None:
            return stored[name][rows].to(F)
        if name not in wide:
            wide[name] = stored[name].to(F)
        return wide[name]

    per = []
    for (old, new), tokens in zip(_requests(case), _tokens(case, cfg.get("vocab_size") or cfg["vocab"], seed)):
        ids = torch.tensor(tokens, device=device)
        last = old + new - 1
        per.append(plain(cfg, T, ids)(slice(last, last + case["steps"] + 1)))
    return [torch.stack([logits[j] for logits in per]) for j in range(case["steps"] + 1)]
