"""The work that this engine is measured on: whole requests through ``Engine.generate``, from the prompts to
the tokens, with the logits of the last step.

Five models, with seeded weights at the shapes that the benchmark uses: LFM2 at 350M and 1.2B (bfloat16), LFM2-350M
in float32, and two models put together from the other parts, Kifetar (windowed sigmoid attention, gated delta rule)
and Minilorn (softmax attention with a sink, attention over compressed rows, matrix memory).  Requests: 1 to 64 of
them, prompts of 1 to 20,001 tokens, alike or ragged, 1 to 128 new tokens each, greedy or sampled.

The weights are drawn so that the most likely token stands out, as a trained model's does: a stream in which
the token's own embedding stays visible, and a head in which every token has a successor.  The tokens of a
run are then the same for every correct implementation, and with them the logits of its last step.
"""
import atexit
import json
import math
import os
import random
import shutil
import tempfile

import torch

from celeg_amd import native
from celeg_amd.engine import Engine
from celeg_amd.sampling import GREEDY, GenerationConfig
from celeg_amd.weights.safetensors_io import write_safetensors

F64 = torch.float64
DEVICE = "cuda" if torch.cuda.is_available() else "cpu"      # (the weights and the 64-bit results; the engine runs on a GPU only)
VOCAB = 65536
STEP_TOKENS = 2048          # most tokens of a step, and of a prompt's portion
MAX_REQUESTS = 64
MAX_CONTEXT = 32768

# ------------------------------------------------------------------------------------------------ models


def _lfm2(hidden, heads, kv_heads, intermediate):
    layers = ["full_attention" if i in (2, 5, 8, 10, 12, 14) else "conv" for i in range(16)]
    return {"architectures": ["Lfm2ForCausalLM"], "model_type": "lfm2", "vocab_size": VOCAB, "hidden_size": hidden,
            "num_hidden_layers": 16, "layer_types": layers, "num_attention_heads": heads, "num_key_value_heads": kv_heads,
            "head_dim": 64, "intermediate_size": intermediate, "block_auto_adjust_ff_dim": False, "rope_theta": 1000000.0,
            "conv_L_cache": 3, "conv_bias": False, "tie_word_embeddings": True, "norm_eps": 1e-5,
            "max_position_embeddings": MAX_CONTEXT, "bos_token_id": 1, "eos_token_id": 7, "pad_token_id": 0}


def _kifetar():
    attention = {"heads": 16, "kv_heads": 8, "dim": 64, "vdim": 64, "scale": 0.125, "mask": {"size": 1024},
                 "rot": {"base": 500000.0, "dims": 32, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
    delta = {"heads": 16, "kv_heads": 8, "dim": 64, "vdim": 64, "conv": 4}
    mlp = {"kind": "dense", "ff": 2048}
    return {"architecture": "Kifetar", "vocab": VOCAB, "width": 1024, "norm": {"eps": 1e-5}, "max_context": 8192,
            "layers": [{"type": "attention", "mixer": attention, "mlp": mlp} if kind == "a" else
                       {"type": "delta", "mixer": delta, "mlp": mlp} for kind in "daadaada"]}


def _minilorn():
    kinds = {"a": ("attention", {"heads": 16, "kv_heads": 8, "dim": 64, "vdim": 64, "scale": 0.125,
                                 "q_temp": {"coef": 0.1, "every": 512}, "softcap": 30.0}),
             "l": ("latent_attention", {"heads": 16, "dim": 64, "rot_dim": 32, "vdim": 64, "q_rank": 512, "kv_rank": 256,
                                        "scale": 96 ** -0.5, "rot": {"base": 500000.0, "dims": 32}, "mask": {"size": 1024}}),
             "m": ("mlstm", {"heads": 8, "dim": 64, "vdim": 128, "gate_cap": 15.0})}
    return {"architecture": "Minilorn", "vocab": VOCAB, "width": 1024, "norm": {"eps": 1e-5}, "max_context": 8192,
            "embedding": {"bigram": {"buckets": 16381, "mul_prev": 7919, "mul_cur": 104729}},
            "layers": [{"type": kinds[c][0], "mixer": kinds[c][1], "mlp": {"kind": "dense", "ff": 3072}} for c in "lmallmal"]}


MODELS = {"lfm2-350m": _lfm2(1024, 16, 8, 4608), "lfm2-1.2b": _lfm2(2048, 32, 8, 8192), "kifetar-1k": _kifetar(), "minilorn-1k": _minilorn()}
# pages of 16 tokens of the cache: 64 requests of 2,112 tokens, or 16 of them beside long ones, for the model that serves
PAGES = {"lfm2-350m": 8704, "lfm2-1.2b": 4096, "kifetar-1k": 4096, "minilorn-1k": 4096}
FLOAT32_PAGES = 1024


def _config(model):
    return MODELS[model]


def _tied(model):
    return model != "minilorn-1k"


def _after(model, token):
    """The token that the head holds for `token`: its partner in a pair, or the next one of a cycle through all."""
    return token ^ 1 if _tied(model) else (token * 5 + 12345) % VOCAB


# Spread of what is written into the residual stream: 32 (LFM2) or 16 sub-layers add about twice the token's own row.
_SPREAD = {"out_proj.weight": 0.0023, "w2.weight": 0.0008, "mix.o": 0.0023, "mlp.down": 0.0008,
           "conv.conv.weight": 0.3, "q.conv": 0.3, "k.conv": 0.3, "v.conv": 0.3, "dt_bias": 1.0, "A_log": 1.0, "i.b": 1.0, "f.b": 2.0,
           "temp": 0.2, "embed_tokens.weight": 0.04, "embed": 0.04, "head": 0.04}


def _weights(model, dtype):
    """{name: tensor} of the checkpoint, drawn on the GPU from a seed of its own per tensor."""
    tied, tensors, signs = _tied(model), {}, None
    for i, e in enumerate(native.describe_config(_config(model))["expected_tensors"]):
        name, shape = e["name"], tuple(e["shape"])
        gen = torch.Generator(device=DEVICE).manual_seed(1000 + i)
        std = next((s for tail, s in _SPREAD.items() if name.endswith(tail)), 0.02)
        if name.endswith(("out_proj.weight", "w2.weight")):
            std *= 1024 / shape[0]
        t = torch.randn(shape, generator=gen, device=DEVICE) * std
        if e["init"] == "around_one":
            t += 1.0
        if name.endswith("_layernorm.weight") or name.endswith(("q.norm", "k.norm")):
            t *= 1.5                                    # queries and keys that prefer some keys to others
        if name.endswith(("norm1b", "norm2b", "norm1b.b", "norm2b.b")):
            t *= 0.025                                  # Kifetar norms what a sub-layer adds: its size is this factor
        tensors[name] = t
    embed = "model.embed_tokens.weight" if tied and model.startswith("lfm2") else "embed"
    table = tensors[embed]
    if tied:
        final = "model.embedding_norm.weight" if model.startswith("lfm2") else "final.norm"
        gen = torch.Generator(device=DEVICE).manual_seed(7)
        signs = torch.randint(0, 2, (table.shape[1],), generator=gen, device=DEVICE) * 2.0 - 1.0
        tensors[final] *= signs
        table[1::2] = table[0::2] * signs
    else:
        order = torch.tensor([_after(model, t) for t in range(VOCAB)], device=DEVICE)
        tensors["head"][order] = table
    return {name: t.to(dtype) for name, t in tensors.items()}


_engines = {}
_checkpoints = []


@atexit.register
def _remove_checkpoints():
    for folder in _checkpoints:
        shutil.rmtree(folder, ignore_errors=True)


def _engine(model, dtype):
    """The program's engine for a model: loaded once, kept for all requests, as a server keeps it."""
    if (model, dtype) not in _engines:
        folder = tempfile.mkdtemp(prefix="celeg_cases_")
        _checkpoints.append(folder)
        with open(os.path.join(folder, "config.json"), "w") as fh:
            json.dump(_config(model), fh)
        weights = {k: v.cpu() for k, v in _weights(model, getattr(torch, dtype)).items()}
        write_safetensors(os.path.join(folder, "model.safetensors"), weights, metadata={"format": "pt"})
        del weights
        torch.cuda.empty_cache()
        context = min(MAX_CONTEXT, _config(model).get("max_context", MAX_CONTEXT))
        _engines[(model, dtype)] = Engine.from_folder(
            folder, dtype=dtype, device="cuda:0", n_pages=FLOAT32_PAGES if dtype == "float32" else PAGES[model], context=context,
            max_active_requests=MAX_REQUESTS, max_batched_tokens=STEP_TOKENS, prefill_chunk_tokens=STEP_TOKENS)
        shutil.rmtree(folder, ignore_errors=True)
    return _engines[(model, dtype)]


# ------------------------------------------------------------------------------------------------ cases


def _case(name, model, requests, low, high, new, sampling="greedy", dtype="bfloat16"):
    case = {"model": model, "dtype": dtype, "requests": requests, "prompt_low": low, "prompt_high": high, "new_tokens": new,
            "sampling": sampling}
    return dict(case, name=name) if name else case


def listed():
    return [
        # the smallest call: a short question, answered with one token (a classifier, a yes or no)
        _case("first_token", "lfm2-350m", 1, 24, 24, 1),
        # one user at an assistant, with the library's default sampling: latency of single tokens
        _case("chat_1", "lfm2-350m", 1, 301, 301, 64, "default"),
        # the headline: eight requests of 2,048 tokens each, decoded together
        _case("batch_8", "lfm2-350m", 8, 2048, 2048, 128),
        # a busy server: 64 requests of all lengths, portions of prompts beside decoding requests, warm sampling
        _case("serve_64", "lfm2-350m", 64, 128, 2048, 64, "warm"),
        # scoring or classifying a document: the prompt alone
        _case("prompt_2048", "lfm2-350m", 1, 2048, 2048, 1),
        # a long document: portions behind up to 18,000 tokens of context
        _case("prompt_20001", "lfm2-350m", 1, 20001, 20001, 1),
        # many short ragged texts classified at once
        _case("prompts_ragged", "lfm2-350m", 24, 5, 401, 1),
        # the wider model: decoding a batch, and prompts
        _case("wide_batch_8", "lfm2-1.2b", 8, 100, 300, 64),
        _case("wide_prompts", "lfm2-1.2b", 3, 1000, 2000, 1),
        # float32, for those who compare with another implementation or debug a checkpoint
        _case("float32_2", "lfm2-350m", 2, 150, 350, 16, "greedy", "float32"),
        # models put together from the other parts: prompts behind a window and a recurrence, then decoding
        _case("kifetar_4", "kifetar-1k", 4, 700, 1500, 32),
        _case("minilorn_4", "minilorn-1k", 4, 700, 1500, 32, "default"),
    ]


def draw(rng):
    def spread(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    model, dtype = rng.choice([("lfm2-350m", "bfloat16")] * 5 + [("lfm2-1.2b", "bfloat16")] * 2 + [("lfm2-350m", "float32")] +
                              [("kifetar-1k", "bfloat16"), ("minilorn-1k", "bfloat16")])
    most, longest, requests_most = {("lfm2-350m", "bfloat16"): (65536, 20001, 64), ("lfm2-1.2b", "bfloat16"): (16384, 16384, 64),
                                    ("lfm2-350m", "float32"): (1024, 1024, 8)}.get((model, dtype), (16384, 8000, 32))
    requests = spread(1, requests_most)
    high = spread(1, min(longest, most // requests))
    low = max(1, int(high * rng.choice([1.0, 0.5, 0.1])))
    new = spread(1, 32 if dtype == "float32" else 128)
    return _case("", model, requests, low, high, new, rng.choice(["greedy", "default", "warm"]), dtype)


def _lengths(case):
    """Prompt lengths between the case's two, spread by the golden ratio: the same for every seed."""
    low, high = case["prompt_low"], case["prompt_high"]
    return [low + int((high - low + 1) * ((i * 0.6180339887) % 1.0)) for i in range(case["requests"])]


SAMPLING = {"greedy": GREEDY, "default": GenerationConfig(), "warm": GenerationConfig(temperature=0.7, top_k=40, top_p=0.9, repetition_penalty=1.0)}


def _prompts(case, seed):
    rng = random.Random(seed)
    return [[rng.randrange(VOCAB) for _ in range(n)] for n in _lengths(case)]


def prepare(case, seed):
    return {"engine": _engine(case["model"], case["dtype"]), "prompts": _prompts(case, seed), "new_tokens": case["new_tokens"],
            "sampling": SAMPLING[case["sampling"]]}


def run(state):
    tokens = state["engine"].generate(state["prompts"], max_new_tokens=state["new_tokens"], generation=state["sampling"], eos_token_ids=[])
    return {"tokens": torch.tensor(tokens), "logits": state["engine"].last_logits}


# ------------------------------------------------------------------------------------------------ work


def _sizes(model):
    """(weights that every token multiplies with, the head's, [(values per key/value row, flops per query and key, window)])."""
    cfg = _config(model)
    body = head = 0
    for e in native.describe_config(cfg)["expected_tensors"]:
        n = math.prod(e["shape"])
        if e["name"] in ("model.embed_tokens.weight", "embed"):
            head = n
        elif e["name"] not in ("bigram", "head"):
            body += n
    rows = []
    if model.startswith("lfm2"):
        hq, hkv = cfg["num_attention_heads"], cfg["num_key_value_heads"]
        rows = [(2 * hkv * 64, 4 * hq * 64, 1 << 30)] * cfg["layer_types"].count("full_attention")
    else:
        for layer in cfg["layers"]:
            m = layer["mixer"]
            window = (m.get("mask") or {}).get("size", 1 << 30)
            if layer["type"] == "attention":
                rows.append((2 * m["kv_heads"] * 64, 4 * m["heads"] * 64, window))
            elif layer["type"] == "latent_attention":
                rows.append((m["kv_rank"] + m["rot_dim"], 2 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), window))
    return body, head, rows


def work(case):
    """Every token's products and attention.  The weights are read once for all prompts and once for every further
    token: no cache of the chip holds them from one step to the next.  A decoded token reads its request's rows."""
    body, head, rows = _sizes(case["model"])
    size = 4 if case["dtype"] == "float32" else 2
    new, lengths = case["new_tokens"], _lengths(case)
    fed = sum(lengths) + len(lengths) * (new - 1)
    flops = 2.0 * body * fed + 2.0 * head * len(lengths) * new
    values = (body + head) * float(new)
    for per_row, per_pair, window in rows:
        for n in lengths:
            last = n + new - 1
            full = min(last, window)
            flops += per_pair * (full * (full + 1) / 2 + (last - full) * window)
            values += per_row * (last + sum(min(t, window) for t in range(n + 1, last + 1)))
    return {"bytes": values * size, "flops": flops}


def tolerance(case):
    """Against 64 bits these paths show 4e-6 in float32 and 0.006 to 0.02 in bfloat16 (16 layers of roundings to 8 bits)."""
    return {"rel": 2e-5, "max": 3e-4} if case["dtype"] == "float32" else {"rel": 0.03, "max": 0.4}


# ------------------------------------------------------------------------------------------------ 64 bits


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _layer_norm(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return _rms(x, w, eps) + b


def _silu(x):
    return x * torch.sigmoid(x)


def _turn(x, angle, neighbours=False):
    """x [n, heads, size], angle [n, pairs]: pair i is the values i and i + pairs, or 2i and 2i + 1; the rest passes."""
    c, s, half = torch.cos(angle)[:, None], torch.sin(angle)[:, None], angle.shape[1]
    if neighbours:
        u, v = x[..., 0::2], x[..., 1::2]
        return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)
    u, v = x[..., :half], x[..., half:2 * half]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * half:]], -1)


def _attend(q, k, v, weigh, window=None):
    """q [n, heads, dim], k and v [n, groups, ..]: `weigh` turns scores [heads, rows, keys] and their mask into weights."""
    n, heads = q.shape[:2]
    group, out = heads // k.shape[1], []
    k, v = k.repeat_interleave(group, 1).permute(1, 2, 0), v.repeat_interleave(group, 1).permute(1, 0, 2)
    block = max(1, int(2e8 // (heads * n)))
    at = torch.arange(n, device=q.device)
    for i in range(0, n, block):
        rows = at[i:i + block, None]
        seen = at[None] <= rows
        if window:
            seen &= rows - at[None] < window
        end = min(i + block, n)
        first = max(0, i - window + 1) if window else 0
        scores = q[i:i + block].permute(1, 0, 2) @ k[:, :, first:end]
        out.append((weigh(scores, seen[:, first:end], rows) @ v[:, first:end]).permute(1, 0, 2))
    return torch.cat(out)


def _softmax(scale):
    return lambda s, seen, rows: torch.softmax((s * scale).masked_fill(~seen, -math.inf), -1)


def _taps(x, w):
    """x [n, channels], w [channels, taps]: the last tap is the row's own."""
    taps = w.shape[1]
    return torch.nn.functional.conv1d(torch.nn.functional.pad(x.T[None], (taps - 1, 0)), w[:, None], groups=x.shape[1])[0].T


def _lfm2_stream(cfg, W, tokens):
    x, eps, n = W["model.embed_tokens.weight"][tokens], cfg["norm_eps"], len(tokens)
    # angles are 32-bit products of position and frequency by definition
    freq = torch.tensor([cfg["rope_theta"] ** (-2.0 * i / 64) for i in range(32)], device=x.device, dtype=torch.float32)
    angle = (torch.arange(n, device=x.device, dtype=torch.float32)[:, None] * freq).to(F64)
    for i, kind in enumerate(cfg["layer_types"]):
        p = f"model.layers.{i}."
        h = _rms(x, W[p + "operator_norm.weight"], eps)
        if kind == "conv":
            b, c, u = (h @ W[p + "conv.in_proj.weight"].T).chunk(3, -1)
            x = x + (c * _taps(b * u, W[p + "conv.conv.weight"][:, 0])) @ W[p + "conv.out_proj.weight"].T
        else:
            p += "self_attn."
            q, k, v = ((h @ W[p + f"{name}_proj.weight"].T).view(n, -1, 64) for name in "qkv")
            q, k = _turn(_rms(q, W[p + "q_layernorm.weight"], eps), angle), _turn(_rms(k, W[p + "k_layernorm.weight"], eps), angle)
            x = x + _attend(q, k, v, _softmax(0.125)).reshape(n, -1) @ W[p + "out_proj.weight"].T
        p = f"model.layers.{i}."
        h = _rms(x, W[p + "ffn_norm.weight"], eps)
        p += "feed_forward."
        x = x + (_silu(h @ W[p + "w1.weight"].T) * (h @ W[p + "w3.weight"].T)) @ W[p + "w2.weight"].T
    return lambda rows: _rms(x[rows], W["model.embedding_norm.weight"], eps) @ W["model.embed_tokens.weight"].T


def _kifetar_mixer(kind, m, h, t, eps):
    n, heads, groups, dim = h.shape[0], m["heads"], m["kv_heads"], m["dim"]
    if kind == "attention":
        q, k = (h @ t["q"].T + t["q.b"]).view(n, heads, dim), (h @ t["k"].T + t["k.b"]).view(n, groups, dim)
        freq, r = [], m["rot"]["scaling"]
        for i in range(m["rot"]["dims"] // 2):
            f = m["rot"]["base"] ** (-2.0 * i / m["rot"]["dims"])
            length = 2.0 * math.pi / f
            share = min(max((r["original"] / length - r["low"]) / (r["high"] - r["low"]), 0.0), 1.0)
            freq.append(share * f + (1.0 - share) * f / r["factor"])
        angle = torch.arange(n, device=h.device, dtype=F64)[:, None] * torch.tensor(freq, device=h.device, dtype=F64)
        turned_q, turned_k = _turn(_rms(q, t["q.norm"], eps), angle), _turn(_rms(k, t["k.norm"], eps), angle)

        def weigh(s, seen, rows):
            return torch.sigmoid(s * (m["scale"] * t["temp"])[:, None, None] + t["pb"][:, None, None]) * seen
        out = _attend(turned_q, turned_k, k, weigh, m["mask"]["size"]) * torch.sigmoid(h @ t["g"].T)[..., None]
        return out.reshape(n, -1) @ t["o"].T
    q, k, v = (_silu(_taps(h @ t[c].T, t[c + ".conv"])).view(n, -1, dim) for c in "qkv")
    q = (q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * dim ** -0.5).repeat_interleave(heads // groups, 1)
    k = (k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(heads // groups, 1)
    beta = torch.sigmoid(h @ t["b"].T)
    decay = torch.exp(-torch.exp(t["A_log"]) * torch.nn.functional.softplus(h @ t["a"].T + t["dt_bias"]))
    state, out = torch.zeros(heads, dim, m["vdim"], device=h.device, dtype=F64), []
    for i in range(n):
        state = state * decay[i, :, None, None]
        state = torch.baddbmm(state, k[i, :, :, None], (beta[i, :, None] * (v[i] - (k[i, :, None] @ state)[:, 0]))[:, None])
        out.append((q[i, :, None] @ state)[:, 0])
    return (_rms(torch.stack(out), t["norm"], eps) * _silu(h @ t["g"].T).view(n, heads, -1)).reshape(n, -1) @ t["o"].T


def _kifetar_stream(cfg, W, tokens):
    x, eps = W["embed"][tokens], cfg["norm"]["eps"]

    def norm(x, name):
        return _layer_norm(x, W[name], W[name + ".b"], eps)
    for i, layer in enumerate(cfg["layers"]):
        p = f"l{i}."
        t = {k[len(p) + 4:]: v for k, v in W.items() if k.startswith(p + "mix.")}
        x = x + norm(_kifetar_mixer(layer["type"], layer["mixer"], norm(x, p + "norm1"), t, eps), p + "norm1b")
        h = norm(x, p + "norm2")
        x = x + norm((_silu(h @ W[p + "mlp.gate"].T) * (h @ W[p + "mlp.up"].T)) @ W[p + "mlp.down"].T, p + "norm2b")
    return lambda rows: norm(x[rows], "final.norm") @ W["embed"].T


def _minilorn_mixer(kind, m, h, t, eps):
    n, heads, dim = h.shape[0], m["heads"], m["dim"]
    at = torch.arange(n, device=h.device)
    if kind == "attention":
        q, k, v = ((h @ t[c].T).view(n, -1, dim) for c in "qkv")
        factor = 1.0 + m["q_temp"]["coef"] * torch.log((at + 1) // m["q_temp"]["every"] + 1.0).to(F64)

        def weigh(s, seen, rows):
            s = (m["softcap"] * torch.tanh(s * m["scale"] / m["softcap"])).masked_fill(~seen, -math.inf)
            sink = t["sink"][:, None, None].expand(-1, s.shape[1], 1)
            return torch.softmax(torch.cat([s, sink], -1), -1)[..., :-1]
        return _attend(q * factor[:, None, None], k, _rms(v, 1.0, eps), weigh).reshape(n, -1) @ t["o"].T
    if kind == "latent_attention":
        rot, rank = m["rot_dim"], m["kv_rank"]
        angle = at.to(F64)[:, None] * torch.tensor([m["rot"]["base"] ** (-2.0 * i / rot) for i in range(rot // 2)], device=h.device, dtype=F64)
        q = (_rms(h @ t["dq"].T, t["dq.norm"], eps) @ t["uq"].T).view(n, heads, dim + rot)
        down = h @ t["dkv"].T
        c = _rms(down[:, :rank], t["dkv.norm"], eps)
        k_turn = _turn(down[:, None, rank:], angle, True).expand(-1, heads, -1)
        q = torch.cat([q[..., :dim], _turn(q[..., dim:], angle, True)], -1)
        k = torch.cat([(c @ t["uk"].T).view(n, heads, dim), k_turn], -1)
        return _attend(q, k, (c @ t["uv"].T).view(n, heads, -1), _softmax(m["scale"]), m["mask"]["size"]).reshape(n, -1) @ t["o"].T
    q, k, v = (h @ t["q"].T).view(n, heads, dim) * dim ** -0.5, (h @ t["k"].T).view(n, heads, dim), (h @ t["v"].T).view(n, heads, -1)
    cap = m["gate_cap"]
    write = cap * torch.tanh((h @ t["i"].T + t["i.b"]) / cap)
    keep = torch.nn.functional.logsigmoid(cap * torch.tanh((h @ t["f"].T + t["f.b"]) / cap))
    # weights of the rows before in closed form: the running maximum only scales numerator and denominator
    total = keep.cumsum(0)
    top = torch.maximum(torch.cummax(write - total, 0).values, torch.zeros_like(total)) + total

    def weigh(s, seen, rows):
        i, j = rows[:, 0], s.shape[-1]
        log = (total[i] - top[i]).T[:, :, None] + (write - total)[:j].T[:, None]
        w = s * torch.exp(log.masked_fill(~seen, -math.inf))
        return w / (torch.maximum(w.sum(-1, keepdim=True).abs(), torch.exp(-top[i]).T[..., None]) + 1e-6)
    out = _rms(_attend(q, k, v, weigh), 1.0, eps).reshape(n, -1)
    return (out * t["norm"] * torch.sigmoid(h @ t["g"].T)) @ t["o"].T


def _minilorn_stream(cfg, W, tokens):
    pair, eps = cfg["embedding"]["bigram"], cfg["norm"]["eps"]
    row = torch.full_like(tokens, pair["buckets"])
    row[1:] = (tokens[:-1] * pair["mul_prev"] + tokens[1:] * pair["mul_cur"]) % pair["buckets"]
    x = W["embed"][tokens] + W["bigram"][row]
    for i, layer in enumerate(cfg["layers"]):
        p = f"l{i}."
        t = {k[len(p) + 4:]: v for k, v in W.items() if k.startswith(p + "mix.")}
        x = x + _minilorn_mixer(layer["type"], layer["mixer"], _rms(x, W[p + "norm1"], eps), t, eps)
        z, act = _rms(x, W[p + "norm2"], eps) @ W[p + "mlp.up"].T, W[p + "mlp.act"]
        right, left = torch.nn.functional.softplus(act[0]), 0.5 + torch.nn.functional.softplus(act[1])
        low = z.clamp(max=0.0)
        x = x + (torch.where(z > 0, right * z * z, left * (torch.expm1(low) - low)) + 0.5 * z) @ W[p + "mlp.down"].T
    return lambda rows: _rms(x[rows], W["final.norm"], eps) @ W["head"].T


def _last_step(case):
    """The requests of the last step, in order: those whose prompts were done last, when every step takes a token of each
    decoding request and then up to STEP_TOKENS of the prompts in order."""
    lengths, new = _lengths(case), case["new_tokens"]
    left, first, step = list(lengths), [None] * len(lengths), 0
    while None in first:
        room = STEP_TOKENS - sum(1 for f in first if f is not None and step < f + new)
        for i, n in enumerate(left):
            part = min(n, room)
            left[i] -= part
            room -= part
            if n and not left[i]:
                first[i] = step
        step += 1
    return [i for i, f in enumerate(first) if f == max(first)]


def exact(case, seed):
    model, new = case["model"], case["new_tokens"]
    stream = {"lfm2": _lfm2_stream, "kife": _kifetar_stream, "mini": _minilorn_stream}[model[:4]]
    W = {k: v.to(F64) for k, v in _weights(model, getattr(torch, case["dtype"])).items()}
    prompts, logits = _prompts(case, seed), []
    for i in _last_step(case):
        tokens = list(prompts[i])
        follow = []
        for _ in range(new):
            follow.append(_after(model, (follow or tokens)[-1]))
        sequence = torch.tensor(tokens + follow[:-1], device=DEVICE)
        scores = stream(_config(model), W, sequence)(slice(len(tokens) - 1, None))
        if scores.argmax(-1).tolist() != follow:
            return None
        logits.append(scores[-1])
    torch.cuda.empty_cache()
    return {"tokens": None, "logits": torch.stack(logits).cpu()}
