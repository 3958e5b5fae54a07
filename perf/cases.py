"""What this engine is timed on: prompts, generation, continuous batching and sampling through its public entry points.

A case is one of four kinds of work, at sizes of the model shapes that ``bench.py`` runs (fewer layers of them, so that a
model is made quickly; a layer's sizes and the vocabulary are whole):

* ``prompt``    a prompt (or two) as one step, the logits behind it (time to the first token);
* ``generate``  prompts in portions of at most 2,048 tokens a step, then tokens one by one for all requests together;
* ``serve``     the same with requests that arrive one after the other: portions of prompts beside decoding requests;
* ``sample``    one token for each row of logits, with the filters and penalties that requests ask for.

The tokens that a request goes on with are given and not sampled (as ``bin/trace_run`` replays them), so that two runs see
the same tokens and every step's logits can be compared.
"""
from __future__ import annotations

import math
import random
from typing import Dict, List, Tuple

import torch

from reinfer_amd.config import config_from_dict
from reinfer_amd.engine import ModelRunner, StepEntry
from reinfer_amd.sampling import Sampler, SamplingParams

BLOCK = 16
PORTION = 2048          # prompt tokens a step, beside the tokens of decoding requests


# ---------------------------------------------------------------------------------------------------------- models
def _qwen3(layers: int, width: int, heads: int, ff: int, tied: bool) -> dict:
    return {"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "num_hidden_layers": layers, "hidden_size": width,
            "num_attention_heads": heads, "num_key_value_heads": 8, "head_dim": 128, "intermediate_size": ff,
            "vocab_size": 151936, "rope_theta": 1000000.0, "rms_norm_eps": 1e-6, "tie_word_embeddings": tied,
            "max_position_embeddings": 16384, "attention_bias": False}


def _puresun() -> dict:
    mixer = {"heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 192, "scale": 192 ** -0.5,
             "mask": {"size": 1024}, "rot": {"base": 10000.0, "dims": 64}}
    mlp = {"kind": "moe", "expert": {"ff": 1536}, "router": {"experts": 16, "top": 4}}
    return {"architecture": "Puresun", "vocab": 32768, "width": 4096, "norm": {"eps": 1e-6}, "logit_softcap": 50.0,
            "embedding": {"bigram": {"buckets": 65521, "mul_prev": 92821, "mul_cur": 689}},
            "layers": [{"type": "latent_attention", "mixer": mixer, "mlp": mlp} for _ in range(3)],
            "loop": {"start": 0, "stop": 1, "times": 2}}


def _kobolix() -> dict:
    memory = {"dim": 128, "gate_cap": 15.0, "heads": 16, "vdim": 256}
    pair = {"left": {"dim": 128, "heads": 32, "kv_heads": 8, "rot": {"base": 1000000.0, "dims": 64}, "scale": 128 ** -0.5,
                     "vdim": 128},
            "right": {"conv": 4, "dim": 128, "heads": 32, "kv_heads": 16, "vdim": 128}}
    dense = {"ff": 11008, "kind": "dense"}
    experts = {"expert": {"ff": 1024}, "kind": "moe", "shared": {"ff": 2048},
               "router": {"experts": 16, "groups": {"count": 4, "keep": 2}, "scale": 2.5, "top": 4}}
    return {"architecture": "Kobolix", "vocab": 32768, "width": 4096, "norm": {"eps": 1e-6}, "residual_mult": 0.5,
            "embedding": {"scale": 8.0},
            "layers": [{"type": "mlstm", "mixer": memory, "mlp": dense}, {"type": "parallel", "mixer": pair, "mlp": experts},
                       {"type": "mlstm", "mixer": memory, "mlp": experts}]}


MODELS = {"qwen3-8b": lambda: _qwen3(8, 4096, 32, 12288, False),
          "qwen3-4b": lambda: _qwen3(8, 2560, 32, 9728, True),
          "qwen3-32b": lambda: _qwen3(4, 5120, 64, 25600, False),
          "puresun": _puresun,
          "kobolix": _kobolix}


def _tensor_shapes(model: str) -> Dict[str, Tuple[int, ...]]:
    """Every tensor of the model, by name."""
    raw, out = MODELS[model](), {}
    if model.startswith("qwen3"):
        h, f, d = raw["hidden_size"], raw["intermediate_size"], raw["head_dim"]
        nq, nkv = raw["num_attention_heads"] * d, raw["num_key_value_heads"] * d
        out["model.embed_tokens.weight"] = (raw["vocab_size"], h)
        for i in range(raw["num_hidden_layers"]):
            p = f"model.layers.{i}."
            a = p + "self_attn."
            out.update({p + "input_layernorm.weight": (h,), a + "q_proj.weight": (nq, h), a + "k_proj.weight": (nkv, h),
                        a + "v_proj.weight": (nkv, h), a + "o_proj.weight": (h, nq), a + "q_norm.weight": (d,),
                        a + "k_norm.weight": (d,), p + "post_attention_layernorm.weight": (h,),
                        p + "mlp.gate_proj.weight": (f, h), p + "mlp.up_proj.weight": (f, h),
                        p + "mlp.down_proj.weight": (h, f)})
        out["model.norm.weight"] = (h,)
        if not raw["tie_word_embeddings"]:
            out["lm_head.weight"] = (raw["vocab_size"], h)
        return out
    h, V = raw["width"], raw["vocab"]
    out["embed"], out["final.norm"] = (V, h), (h,)
    for i, L in enumerate(raw["layers"]):
        p, m, f = f"l{i}.", L["mixer"], L["mlp"]
        out[p + "norm1"] = (h,)
        if L["type"] == "latent_attention":
            H, D, R, Dv, r = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
            out.update({p + "mix.q": (H * (D + R), h), p + "mix.dkv": (r + R, h), p + "mix.dkv.norm": (r,),
                        p + "mix.uk": (H * D, r), p + "mix.uv": (H * Dv, r), p + "mix.g": (H * Dv, h),
                        p + "mix.o": (h, H * Dv)})
        elif L["type"] == "mlstm":
            H, D, Dv = m["heads"], m["dim"], m["vdim"]
            out.update({p + "mix.q": (H * D, h), p + "mix.k": (H * D, h), p + "mix.v": (H * Dv, h), p + "mix.g": (H * Dv, h),
                        p + "mix.o": (h, H * Dv), p + "mix.norm": (H * Dv,), p + "mix.i": (H, h), p + "mix.i.b": (H,),
                        p + "mix.f": (H, h), p + "mix.f.b": (H,)})
        else:
            a, b = m["left"], m["right"]
            q = p + "mix.left."
            out.update({q + "q": (a["heads"] * a["dim"], h), q + "k": (a["kv_heads"] * a["dim"], h),
                        q + "v": (a["kv_heads"] * a["vdim"], h), q + "o": (h, a["heads"] * a["vdim"]), q + "out": (h,)})
            q, nk, nv = p + "mix.right.", b["kv_heads"] * b["dim"], b["heads"] * b["vdim"]
            out.update({q + "q": (nk, h), q + "k": (nk, h), q + "v": (nv, h), q + "q.conv": (nk, b["conv"]),
                        q + "k.conv": (nk, b["conv"]), q + "v.conv": (nv, b["conv"]), q + "b": (b["heads"], h),
                        q + "a": (b["heads"], h), q + "A_log": (b["heads"],), q + "dt_bias": (b["heads"],),
                        q + "norm": (b["vdim"],), q + "g": (nv, h), q + "o": (h, nv), q + "out": (h,)})
        gated = model == "kobolix"
        if gated:
            out[p + "norm2"] = (h,)
        if f["kind"] == "dense":
            out.update({p + "mlp.gate": (f["ff"], h), p + "mlp.up": (f["ff"], h), p + "mlp.down": (h, f["ff"])})
            continue
        out[p + "mlp.router"] = (f["router"]["experts"], h)
        parts = [(f"e{e}.", f["expert"]["ff"]) for e in range(f["router"]["experts"])]
        for name, ff in parts + ([("shared.", f["shared"]["ff"])] if f.get("shared") else []):
            if gated:
                out[p + "mlp." + name + "gate"] = (ff, h)
            out[p + "mlp." + name + "up"], out[p + "mlp." + name + "down"] = (ff, h), (h, ff)
    if model == "puresun":
        out.update({"bigram": (raw["embedding"]["bigram"]["buckets"] + 1, h), "loop.step": (raw["loop"]["times"], h),
                    "head": (V, h)})
    return out


def _weights(model: str, seed: int, dtype: torch.dtype) -> Dict[str, torch.Tensor]:
    """Random weights: matrices of deviation 0.02, norms around one (around zero where a design stores them so), gate biases
    and decays over the range that such layers are initialised to (a memory of a few to some hundred tokens). Where there
    are experts, a token's embedding leans towards the experts that are its own, and layers add little to the stream: the
    routers then choose clearly, as trained ones do, and not by the last bit of near ties."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(shape, lo, hi):
        return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo

    out = {}
    for name, shape in _tensor_shapes(model).items():
        last = name.rsplit(".", 1)[-1]
        if name.endswith(".f.b"):
            t = uniform(shape, 2.0, 6.0)
        elif name.endswith(".i.b"):
            t = uniform(shape, -1.0, 1.0)
        elif last == "A_log":
            t = torch.log(uniform(shape, 1.0, 16.0))
        elif last == "dt_bias":
            dt = torch.exp(uniform(shape, math.log(1e-3), math.log(1e-1)))
            t = dt + torch.log(-torch.expm1(-dt))
        elif last == "conv":
            t = uniform(shape, -0.5, 0.5)
        elif len(shape) == 1:
            offset = model == "kobolix" and (last in ("norm1", "norm2") or name == "final.norm")
            t = uniform(shape, -0.2, 0.2) if offset else uniform(shape, 0.8, 1.2)
        else:
            adds = not model.startswith("qwen3") and (last in ("down", "o"))
            t = torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, 0.005 if adds else 0.02, generator=g)
        out[name] = t.to(dtype)
    if not model.startswith("qwen3"):
        raw = MODELS[model]()
        x = torch.randn(out["embed"].shape, generator=g, device="cuda")
        for i, L in enumerate(raw["layers"]):
            if "router" in L["mlp"]:
                r = L["mlp"]["router"]
                groups = r.get("groups") or {"count": 1, "keep": 1}
                size, n = r["experts"] // groups["count"], r["top"] // groups["keep"]
                own = torch.rand((len(x), groups["count"], size), generator=g, device="cuda")
                own = own >= own.topk(n, -1)[0][..., -1:]
                kept = torch.rand((len(x), groups["count"]), generator=g, device="cuda")
                own &= (kept >= kept.topk(groups["keep"], -1)[0][:, -1:])[..., None]
                x += 4.0 * own.flatten(1).float() @ out[f"l{i}.mlp.router"].float()
        out["embed"] = (x / raw["embedding"].get("scale", 1.0)).to(dtype)
    return out


# ----------------------------------------------------------------------------------------------------------- steps
def _lengths(case: dict) -> List[int]:
    """The prompts' lengths: spread evenly over the case's range, in a mixed order."""
    n, lo, hi = case["requests"], case["shortest"], case["longest"]
    out = [lo + (hi - lo) * i // max(1, n - 1) for i in range(n)] if n > 1 else [hi]
    random.Random(n * 1000003 + hi).shuffle(out)
    return out


def _steps(case: dict) -> List[List[Tuple[int, int, int, bool]]]:
    """The steps of a pass: each a list of (request, first token, tokens, whether the last one's logits are wanted)."""
    lengths = _lengths(case)
    if case["kind"] == "prompt":
        return [[(i, 0, n, True) for i, n in enumerate(lengths)]]
    new, done = case["new"], [0] * len(lengths)
    steps = []
    while any(d < n + new for d, n in zip(done, lengths)):
        entries, left = [], PORTION
        prompts = [i for i, n in enumerate(lengths) if done[i] < n]
        if case["kind"] == "serve" or not prompts:
            for i, n in enumerate(lengths):
                if n <= done[i] < n + new:
                    entries.append((i, done[i], 1, True))
        if case["kind"] == "serve":
            prompts = prompts[:1]       # one request arrives a step, or goes on with its prompt
        for i in prompts:
            take = min(left, lengths[i] - done[i])
            if take > 0:
                entries.append((i, done[i], take, done[i] + take == lengths[i]))
                left -= take
        for i, _, take, _ in entries:
            done[i] += take
        steps.append(entries)
    return steps


def _tokens(case: dict, seed: int) -> List[List[int]]:
    vocab = _vocab(case["model"])
    g = torch.Generator().manual_seed(seed + 77)
    return [torch.randint(0, vocab, (n + case["new"],), generator=g).tolist() for n in _lengths(case)]


def _vocab(model: str) -> int:
    raw = MODELS[model]()
    return raw["vocab_size"] if model.startswith("qwen3") else raw["vocab"]


# ------------------------------------------------------------------------------------------------------- sampling
def _sampling(case: dict, seed: int):
    """Logits of a peaked distribution (a few likely tokens over a bell of unlikely ones), each row's options in turn, and
    the tokens that its request holds so far."""
    n, V = case["rows"], case["vocab"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    logits = torch.randn((n, V), generator=g, device="cuda") * 2.5
    r = random.Random(seed)
    params, history = [], []
    for i in range(n):
        k = i % 4
        params.append(SamplingParams(
            temperature=(0.7, 1.0, 0.6, 0.8)[k], top_k=(None, 50, 20, None)[k], top_p=(0.9, None, 0.95, None)[k],
            min_p=0.05 if k == 3 else None, repeat_penalty=1.1 if k == 2 else None,
            presence_penalty=0.5 if k == 3 else None, seed=r.getrandbits(40), max_tokens=16))
        history.append([r.randrange(V) for _ in range(case["history"])])
    return logits, params, [p.seed for p in params], [len(h) for h in history], history


# ----------------------------------------------------------------------------------------------------------- cases
def _prompt(name, model, longest, requests=1, shortest=None, dtype="bfloat16"):
    return {"name": name, "kind": "prompt", "model": model, "dtype": dtype, "requests": requests,
            "shortest": shortest or longest, "longest": longest, "new": 0}


def _generate(name, model, requests, shortest, longest, new, dtype="bfloat16", kind="generate"):
    return {"name": name, "kind": kind, "model": model, "dtype": dtype, "requests": requests, "shortest": shortest,
            "longest": longest, "new": new}


def listed() -> List[dict]:
    return [
        # one user's chat turn: a short question and its answer, where every launch counts
        _generate("chat turn", "qwen3-8b", 1, 53, 53, 32),
        # a handful of users with a page of context each: the shape of the headline figure
        _generate("eight users", "qwen3-8b", 8, 512, 1536, 32),
        # a busy server between two arrivals: many short contexts
        _generate("full server", "qwen3-4b", 48, 40, 400, 24),
        # the first token of a short question, of a page, and of a long document through the widest layers
        _prompt("short prompt", "qwen3-8b", 97),
        _prompt("page prompt", "qwen3-8b", 1733),
        _prompt("long prompt", "qwen3-32b", 7901),
        # continuous batching: prompts arrive while other requests decode
        _generate("arrivals", "qwen3-4b", 12, 60, 1500, 16, kind="serve"),
        # the 32-bit path, which other implementations are checked against
        _generate("32-bit", "qwen3-4b", 4, 60, 500, 12, dtype="float32"),
        # a mixture of experts over a cached latent: a prompt
        _prompt("expert prompt", "puresun", 1900),
        # recurrent memories beside attention, and gated experts: prompts, and a handful of users
        _prompt("memory prompt", "kobolix", 1219, requests=2, shortest=640),
        _generate("memory users", "kobolix", 8, 100, 300, 32),
        # the next tokens of a batch whose requests ask for filters and penalties
        {"name": "filtered sampling", "kind": "sample", "rows": 24, "vocab": 151936, "history": 300},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["prompt", "prompt", "generate", "generate", "serve", "32-bit", "design", "design", "sample"])
    if kind == "prompt":
        model = rng.choice(["qwen3-8b", "qwen3-4b", "qwen3-32b"])
        out = _prompt("", model, _log_int(rng, 16, 7000 if model == "qwen3-32b" else 8000))
    elif kind in ("generate", "serve"):
        n, hi = _log_int(rng, 1, 64), _log_int(rng, 40, 1800)
        hi = min(hi, 12000 // n)
        out = _generate("", rng.choice(["qwen3-8b", "qwen3-4b"]), n, _log_int(rng, 16, hi) if hi > 16 else hi, hi,
                        rng.randint(8, 32), kind=kind)
        if kind == "serve":
            out["requests"] = min(n, 16)
            out["new"] = rng.randint(8, 16)
    elif kind == "32-bit":
        hi = _log_int(rng, 20, 600)
        out = _generate("", "qwen3-4b", rng.randint(1, 4), _log_int(rng, 10, hi), hi, rng.randint(4, 12), dtype="float32")
    elif kind == "design":
        model = rng.choice(["puresun", "kobolix"])
        if rng.random() < 0.5:
            hi = _log_int(rng, 30, 2000)
            out = _prompt("", model, hi, rng.choice([1, 1, 2]), max(16, hi // rng.randint(1, 3)))
        else:
            hi = _log_int(rng, 30, 400)
            out = _generate("", model, _log_int(rng, 1, 24), max(16, hi // rng.randint(1, 3)), hi, rng.randint(8, 32))
    else:
        return {"kind": "sample", "rows": _log_int(rng, 1, 64), "vocab": rng.choice([32768, 151936]),
                "history": _log_int(rng, 1, 4000)}
    del out["name"]
    return out


def prepare(case: dict, seed: int) -> dict:
    if case["kind"] == "sample":
        logits, params, seeds, positions, history = _sampling(case, seed)
        return {"sampler": Sampler(logits.device), "logits": logits, "options": (params, seeds, positions, history)}
    dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    tokens = _tokens(case, seed)
    blocks = sum(-(-len(t) // BLOCK) + 1 for t in tokens)
    runner = ModelRunner.from_config(config_from_dict(MODELS[case["model"]]()), dtype=case["dtype"],
                                     weights=_weights(case["model"], seed, dtype), block_size=BLOCK,
                                     num_blocks=blocks + 8, max_seqs=max(16, case["requests"]),
                                     max_model_len=max(len(t) for t in tokens) + BLOCK)
    steps = [[(i, tokens[i][at:at + n], [n - 1] if want else []) for i, at, n, want in entries] for entries in _steps(case)]
    return {"runner": runner, "requests": list(range(len(tokens))), "steps": steps}


def run(state: dict):
    if "sampler" in state:
        return state["sampler"].sample(state["logits"], *state["options"])
    runner, out = state["runner"], []
    for rid in state["requests"]:
        runner.add_request(rid)
    for entries in state["steps"]:
        logits = runner.step([StepEntry(rid, tokens, want) for rid, tokens, want in entries])
        if logits.shape[0]:
            out.append(logits.clone())          # the next step writes over its buffer
    for rid in state["requests"]:
        runner.free_request(rid)
    return torch.cat(out)


# ------------------------------------------------------------------------------------------------------------ work
def _layer_work(model: str):
    """(matrix elements that every token goes through, elements of one expert, experts, chosen) a layer run, and the bytes
    that a cached token takes a layer over the element size."""
    raw, shapes = MODELS[model](), _tensor_shapes(model)
    out = []
    if model.startswith("qwen3"):
        for i in range(raw["num_hidden_layers"]):
            p = f"model.layers.{i}."
            out.append((sum(math.prod(s) for n, s in shapes.items() if n.startswith(p)), 0, 0, 0,
                        2 * raw["num_key_value_heads"] * raw["head_dim"], raw["num_attention_heads"] * raw["head_dim"], 0))
        return out
    loop = raw.get("loop")
    order = list(range(len(raw["layers"])))
    if loop:
        a, b = loop["start"], loop["stop"]
        order = order[:a] + order[a:b] * loop["times"] + order[b:]
    for i in order:
        p, L = f"l{i}.", raw["layers"][i]
        mine = {n: math.prod(s) for n, s in shapes.items() if n.startswith(p)}
        expert = sum(v for n, v in mine.items() if n.startswith(p + "mlp.e0."))
        rest = sum(v for n, v in mine.items() if not n.startswith(p + "mlp.e"))
        router = L["mlp"].get("router", {"experts": 0, "top": 0})
        m = L["mixer"]
        if L["type"] == "latent_attention":
            cache, heads = m["kv_rank"] + m["rot_dim"], m["heads"] * (m["dim"] + m["rot_dim"])
            out.append((rest, expert, router["experts"], router["top"], cache, heads, m["mask"]["size"]))
        elif L["type"] == "mlstm":
            out.append((rest, expert, router["experts"], router["top"], 0, 0, 0))
        else:
            a = m["left"]
            out.append((rest, expert, router["experts"], router["top"], 2 * a["kv_heads"] * a["dim"], a["heads"] * a["dim"], 0))
    return out


def work(case: dict) -> dict:
    """Bytes: each step reads every weight that its tokens meet once (experts: as many as its choices are expected to name),
    the keys and values its queries see once, and writes its logits; flops: every token through its own weights and keys."""
    if case["kind"] == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": 4 * n, "flops": 4 * n}
    size = 4 if case["dtype"] == "float32" else 2
    raw = MODELS[case["model"]]()
    head = _vocab(case["model"]) * (raw["hidden_size"] if "hidden_size" in raw else raw["width"])
    width = head // _vocab(case["model"])
    layers = _layer_work(case["model"])
    total, flops = 0.0, 0.0
    for entries in _steps(case):
        T = sum(n for _, _, n, _ in entries)
        wanted = sum(1 for e in entries if e[3])
        total += size * (T * width + (head if wanted else 0)) + 4 * wanted * _vocab(case["model"])
        flops += 2.0 * wanted * head
        for dense, expert, experts, top, cache, q, window in layers:
            met = experts * (1.0 - (1.0 - top / experts) ** T) if experts else 0.0
            total += size * (dense + met * expert)
            flops += 2.0 * T * (dense + top * expert)
            for _, at, n, _ in entries:
                seen = at + n if not window else min(at + n, window + n)
                total += size * cache * seen
                mean = at + 0.5 * (n + 1)
                flops += 4.0 * q * n * (min(mean, window) if window else mean)
    return {"bytes": total, "flops": flops}


def tolerance(case: dict):
    if case["kind"] == "sample":
        return "exact"
    # against 64 bits the 32-bit path is off by 9e-6, bfloat16 by 0.014 to 0.019 over random layers that each change the whole
    # stream, and by 0.002 to 0.003 where layers add little to it
    if case["dtype"] == "float32":
        return {"rel": 4e-5, "max": 6e-4}
    return {"rel": 0.03, "max": 0.3} if case["model"].startswith("qwen3") else {"rel": 0.01, "max": 0.1}


# ----------------------------------------------------------------------------------------------------------- exact
D = torch.float64


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _turn(x, dims, base, neighbours):
    """x [T, heads, d]: pairs of the first ``dims`` entries (a half apart, or neighbours) turned by p base^(-2i/dims)."""
    i = torch.arange(dims // 2, dtype=D, device=x.device)
    a = torch.arange(x.shape[0], dtype=D, device=x.device)[:, None] * (float(base) ** (-2.0 * i / dims))[None]
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    out = x.clone()
    one = slice(0, dims, 2) if neighbours else slice(0, dims // 2)
    two = slice(1, dims, 2) if neighbours else slice(dims // 2, dims)
    out[..., one], out[..., two] = x[..., one] * c - x[..., two] * s, x[..., two] * c + x[..., one] * s
    return out


def _attend(q, k, v, scale, window=0):
    """q [T, H, d], k, v [T, G, d]: head by head, queries in runs."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
    j = torch.arange(T, device=q.device)[None]
    for lo in range(0, T, 2048):
        i = torch.arange(lo, min(T, lo + 2048), device=q.device)[:, None]
        hidden = (j > i) if not window else (j > i) | (i - j >= window)
        for h in range(H):
            kk, vv = k[:, h * G // H].contiguous(), v[:, h * G // H].contiguous()
            s = (q[lo:lo + 2048, h] @ kk.t().contiguous()) * scale
            out[lo:lo + 2048, h] = torch.softmax(s.masked_fill_(hidden, float("-inf")), -1) @ vv
    return out.reshape(T, -1)


def _qwen3_exact(w, raw, ids, wanted):
    eps, d = raw["rms_norm_eps"], raw["head_dim"]
    x = w["model.embed_tokens.weight"][ids].to(D)
    for n in range(raw["num_hidden_layers"]):
        p = f"model.layers.{n}."
        a = {k[len(p):-7]: t.to(D) for k, t in w.items() if k.startswith(p)}
        h = _rms(x, eps) * a["input_layernorm"]
        q, k, v = ((h @ a[f"self_attn.{c}_proj"].t()).view(len(ids), -1, d) for c in "qkv")
        q = _turn(_rms(q, eps) * a["self_attn.q_norm"], d, raw["rope_theta"], False)
        k = _turn(_rms(k, eps) * a["self_attn.k_norm"], d, raw["rope_theta"], False)
        x = x + _attend(q, k, v, d ** -0.5) @ a["self_attn.o_proj"].t()
        h = _rms(x, eps) * a["post_attention_layernorm"]
        x = x + (_silu(h @ a["mlp.gate_proj"].t()) * (h @ a["mlp.up_proj"].t())) @ a["mlp.down_proj"].t()
    y = _rms(x[wanted], eps) * w["model.norm.weight"].to(D)
    head = w["model.embed_tokens.weight" if raw["tie_word_embeddings"] else "lm_head.weight"]
    return torch.cat([y @ part.to(D).t() for part in head.split(16384)], -1)


def _experts(h, a, share, gated):
    """sum over experts of share [T, E] times the expert's result, each over the rows that chose it."""
    out = torch.zeros_like(h)
    for e in range(share.shape[1]):
        rows = share[:, e].nonzero()[:, 0]
        if len(rows):
            g, p = h[rows], f"mlp.e{e}."
            u = _silu(g @ a[p + "gate"].t()) * (g @ a[p + "up"].t()) if gated else torch.relu(g @ a[p + "up"].t()) ** 2
            out[rows] += share[rows, e, None] * (u @ a[p + "down"].t())
    return out


def _layer_tensors(w, i):
    p = f"l{i}."
    return {k[len(p):]: t.to(D) for k, t in w.items() if k.startswith(p)}


def _puresun_exact(w, raw, ids, wanted):
    eps, b, loop = raw["norm"]["eps"], raw["embedding"]["bigram"], raw["loop"]
    rows = torch.full_like(ids, b["buckets"])
    rows[1:] = (ids[:-1] * b["mul_prev"] + ids[1:] * b["mul_cur"]) % b["buckets"]
    x = w["embed"][ids].to(D) + w["bigram"][rows].to(D)
    first, T = x.clone(), len(ids)
    runs = [(i, t) for t in range(loop["times"]) for i in range(loop["start"], loop["stop"])]
    runs = [(i, None) for i in range(loop["start"])] + runs + [(i, None) for i in range(loop["stop"], len(raw["layers"]))]
    for i, t in runs:
        if t is not None and i == loop["start"]:
            x = x + (first if t else 0.0) + w["loop.step"][t].to(D)
        a, m, r = _layer_tensors(w, i), raw["layers"][i]["mixer"], raw["layers"][i]["mlp"]["router"]
        H, dim, R, rank = m["heads"], m["dim"], m["rot_dim"], m["kv_rank"]
        h = _rms(x, eps) * a["norm1"]
        q, down = (h @ a["mix.q"].t()).view(T, H, dim + R), h @ a["mix.dkv"].t()
        c = _rms(down[:, :rank], eps) * a["mix.dkv.norm"]
        kr = _turn(down[:, None, rank:], R, m["rot"]["base"], False).expand(T, H, R)
        q = torch.cat([q[..., :dim], _turn(q[..., dim:], R, m["rot"]["base"], False)], -1)
        k = torch.cat([(c @ a["mix.uk"].t()).view(T, H, dim), kr], -1)
        o = _attend(q, k, (c @ a["mix.uv"].t()).view(T, H, -1), m["scale"], m["mask"]["size"])
        y = (o * torch.sigmoid(h @ a["mix.g"].t())) @ a["mix.o"].t()
        val, idx = torch.topk(h @ a["mlp.router"].t(), r["top"], dim=-1)
        share = torch.zeros(T, r["experts"], dtype=D, device=x.device).scatter_(1, idx, torch.softmax(val, -1))
        x = x + y + _experts(h, a, share, False)
    y = (_rms(x[wanted], eps) * w["final.norm"].to(D)) @ w["head"].to(D).t()
    return raw["logit_softcap"] * torch.tanh(y / raw["logit_softcap"])


def _matrix_memory(h, a, m, eps):
    H, dk, dv, cap, T = m["heads"], m["dim"], m["vdim"], m["gate_cap"], h.shape[0]
    q, k, v = ((h @ a["mix." + c].t()).view(T, H, -1) for c in "qkv")
    q = q * dk ** -0.5
    gi = cap * torch.tanh((h @ a["mix.i"].t() + a["mix.i.b"]) / cap)
    gf = torch.nn.functional.logsigmoid(cap * torch.tanh((h @ a["mix.f"].t() + a["mix.f.b"]) / cap))
    S, n, top = (torch.zeros(s, dtype=D, device=h.device) for s in ((H, dk, dv), (H, dk), (H,)))
    out = torch.empty(T, H, dv, dtype=D, device=h.device)
    for t in range(T):
        new = torch.maximum(gf[t] + top, gi[t])
        keep, take = torch.exp(gf[t] + top - new)[:, None], torch.exp(gi[t] - new)[:, None]
        tk, top = take * k[t], new
        S.mul_(keep[..., None]).add_(tk[..., None] * v[t][:, None])
        n.mul_(keep).add_(tk)
        den = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
        out[t] = (S * q[t][..., None]).sum(1) / den[:, None]
    o = _rms(out, eps).reshape(T, -1) * a["mix.norm"]
    return (o * torch.sigmoid(h @ a["mix.g"].t())) @ a["mix.o"].t()


def _delta_rule(h, a, p, m, eps):
    H, G, dk, T = m["heads"], m["kv_heads"], m["dim"], h.shape[0]

    def filtered(c):
        x, f = h @ a[p + c].t(), a[p + c + ".conv"]
        x = torch.cat([x.new_zeros(f.shape[1] - 1, x.shape[1]), x])
        return _silu(sum(x[j:j + T] * f[:, j] for j in range(f.shape[1])))
    q, k, v = filtered("q").view(T, G, dk), filtered("k").view(T, G, dk), filtered("v").view(T, H, -1)
    q = (q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * dk ** -0.5).repeat_interleave(H // G, 1)
    k = (k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
    beta = torch.sigmoid(h @ a[p + "b"].t())
    decay = torch.exp(-torch.exp(a[p + "A_log"]) * torch.nn.functional.softplus(h @ a[p + "a"].t() + a[p + "dt_bias"]))
    S = torch.zeros(H, dk, v.shape[2], dtype=D, device=h.device)
    out = torch.empty(T, H, v.shape[2], dtype=D, device=h.device)
    for t in range(T):
        S.mul_(decay[t][:, None, None])
        u = beta[t][:, None] * (v[t] - (S * k[t][..., None]).sum(1))
        S.add_(k[t][..., None] * u[:, None])
        out[t] = (S * q[t][..., None]).sum(1)
    o = (_rms(out, eps) * a[p + "norm"]).reshape(T, -1)
    return (o * _silu(h @ a[p + "g"].t())) @ a[p + "o"].t()


def _kobolix_exact(w, raw, ids, wanted):
    eps, mult, T = raw["norm"]["eps"], raw["residual_mult"], len(ids)
    x = w["embed"][ids].to(D) * raw["embedding"]["scale"]
    for i, L in enumerate(raw["layers"]):
        a, m, f = _layer_tensors(w, i), L["mixer"], L["mlp"]
        h = _rms(x, eps) * (1.0 + a["norm1"])
        if L["type"] == "mlstm":
            y = _matrix_memory(h, a, m, eps)
        else:
            c, rot = m["left"], m["left"]["rot"]
            q, k = (_turn((h @ a["mix.left." + s].t()).view(T, -1, c["dim"]), rot["dims"], rot["base"], True) for s in "qk")
            v = (h @ a["mix.left.v"].t()).view(T, -1, c["vdim"])
            left = _attend(q, k, v, c["scale"]) @ a["mix.left.o"].t()
            right = _delta_rule(h, a, "mix.right.", m["right"], eps)
            y = 0.5 * (_rms(left, eps) * a["mix.left.out"] + _rms(right, eps) * a["mix.right.out"])
        x = x + mult * y
        h = _rms(x, eps) * (1.0 + a["norm2"])
        if f["kind"] == "dense":
            y = (_silu(h @ a["mlp.gate"].t()) * (h @ a["mlp.up"].t())) @ a["mlp.down"].t()
        else:
            r = f["router"]
            s, size = torch.sigmoid(h @ a["mlp.router"].t()), r["experts"] // r["groups"]["count"]
            best = torch.topk(s.view(T, -1, size).topk(2, -1)[0].sum(-1), r["groups"]["keep"], -1)[1]
            kept = torch.zeros(T, r["groups"]["count"], dtype=torch.bool, device=x.device).scatter_(1, best, True)
            val, idx = torch.topk(s.masked_fill(~kept.repeat_interleave(size, 1), -1.0), r["top"], -1)
            share = torch.zeros_like(s).scatter_(1, idx, val * r["scale"])
            y = _experts(h, a, share, True)
            y = y + (_silu(h @ a["mlp.shared.gate"].t()) * (h @ a["mlp.shared.up"].t())) @ a["mlp.shared.down"].t()
        x = x + mult * y
    return (_rms(x[wanted], eps) * (1.0 + w["final.norm"].to(D))) @ w["embed"].to(D).t()


def exact(case: dict, seed: int):
    if case["kind"] == "sample":
        return None
    dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    model, raw = case["model"], MODELS[case["model"]]()
    w, tokens, steps = _weights(model, seed, dtype), _tokens(case, seed), _steps(case)
    forward = {"puresun": _puresun_exact, "kobolix": _kobolix_exact}.get(model, _qwen3_exact)
    at = {}                 # request -> its wanted positions, in order
    for i, lo, n, want in (e for entries in steps for e in entries):
        if want:
            at.setdefault(i, []).append(lo + n - 1)
    rows = {}
    for i, wanted in at.items():
        ids = torch.tensor(tokens[i], dtype=torch.long, device="cuda")[:wanted[-1] + 1]
        got = forward(w, raw, ids, torch.tensor(wanted, device="cuda"))
        rows.update({(i, p): got[k] for k, p in enumerate(wanted)})
    return torch.stack([rows[i, lo + n - 1] for entries in steps for i, lo, n, want in entries if want])
