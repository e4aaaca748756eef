"""Attention kernels for single tokens against the tile kernels that take them otherwise, called as the host code calls them:
the same bits where they are claimed (attention with biases), no larger distance from 64 bits elsewhere (sigmoid weights)."""
import ctypes
import json
import math

import pytest
import torch

from celeg_amd import native
from helpers import EngineDriver

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16
PAGE = 16


def check(code):
    assert code == 0, f"error {code}"


def ptr(t):
    return ctypes.c_void_p(t.data_ptr() if t is not None else None)


def ints(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


class Decoding:
    """One new token of every request: `contexts` says how many keys each has, its own among them."""

    def __init__(self, contexts, H, G, D, V, layers=2, layer=1, seed=1, spread=1.0):
        gen = torch.Generator().manual_seed(seed)
        r = lambda *s: torch.randn(*s, generator=gen)
        n, per = len(contexts), (max(contexts) + PAGE - 1) // PAGE
        pages = torch.randperm(n * per, generator=gen).int().view(n, per)
        self.sizes, self.layers, self.layer, self.contexts = (H, G, D, V), layers, layer, contexts
        self.k, self.v = r(n * per, layers, G, PAGE, D).to(BF).to(DEV), (r(n * per, layers, G, V, PAGE) + 0.3).to(BF).to(DEV)
        # what lies behind a request's last key may be anything
        for i, c in enumerate(contexts):
            if c % PAGE:
                page = int(pages[i, c // PAGE])
                self.k[page, :, :, c % PAGE:] = float("nan")
                self.v[page, :, :, :, c % PAGE:] = float("nan")
        self.q = (spread * r(n, H * D)).to(BF).to(DEV)
        self.slots = ints([(i + 1) % n for i in range(n)])
        table = torch.empty_like(pages)
        for i in range(n):
            table[(i + 1) % n] = pages[i]
        self.pages, self.table = pages, table.to(DEV)
        self.positions, self.cu = ints([c - 1 for c in contexts]), ints(list(range(n + 1)))
        self.n, self.per = n, per

    def keys_and_values(self, i):
        """of request i: [keys, G, D] and [keys, G, V], 64-bit"""
        at, c = self.pages[i].long().to(DEV), self.contexts[i]
        k = self.k[at, self.layer].double().permute(0, 2, 1, 3).reshape(-1, self.sizes[1], self.sizes[2])[:c]
        v = self.v[at, self.layer].double().permute(0, 3, 1, 2).reshape(-1, self.sizes[1], self.sizes[3])[:c]
        return k, v


BIASED = [  # heads, kv heads, numbers of a key, of a value
    (16, 8, 64, 64), (16, 1, 32, 96), (4, 2, 96, 40), (3, 3, 128, 128), (6, 2, 64, 128), (16, 1, 32, 128), (8, 2, 48, 24)]
OPTIONS = {
    "plain": {}, "window": dict(window=129), "window and kept keys": dict(window=70, keep_first=66), "one": dict(sink_one=1),
    "sink and cap": dict(sink=True, softcap=30.0), "bias": dict(bias=True, gate=True),
    "all": dict(bias=True, gate=True, sink=True, softcap=5.0, coef=0.3, every=64, window=513, keep_first=3),
    "temperature": dict(coef=0.1, every=512, sink=True, softcap=30.0)}


@pytest.mark.parametrize("option", list(OPTIONS))
@pytest.mark.parametrize("H,G,D,V", BIASED)
def test_biased_attention_of_single_tokens_has_the_tiles_bits(H, G, D, V, option):
    o = OPTIONS[option]
    contexts = [1, 64, 65, 700, 513, 1100, 16, 129, 577]
    case = Decoding(contexts, H, G, D, V, seed=D + V, spread=1.5)
    gen = torch.Generator().manual_seed(7)
    heads = lambda size: (size * torch.randn(H, generator=gen)).to(DEV)
    r1, r2, sink = heads(0.3), heads(0.01).abs(), heads(1.0)
    gate = torch.randn(case.n, H * V, generator=gen).to(BF).to(DEV)
    got = {}
    for form in (0, 2):
        out = torch.full((case.n, H * V), float("nan"), dtype=BF, device=DEV)
        check(native.lib().celeg_biased_attention_fast(
            form, ptr(case.q), H * D, ptr(case.k), ptr(case.v), ptr(case.table), case.per, ptr(case.cu), ptr(case.slots), ptr(case.positions),
            case.n, case.n, ptr(r1 if o.get("bias") else None), ptr(r2 if o.get("bias") else None), ptr(gate if o.get("gate") else None), H * V,
            ptr(out), H * V, H, G, D, V, PAGE, case.layers, case.layer, ctypes.c_float(D ** -0.5), ctypes.c_float(o.get("coef", 0.0)),
            o.get("every", 1), o.get("window", 0), o.get("keep_first", 0), o.get("sink_one", 0), ptr(sink if o.get("sink") else None),
            ctypes.c_float(o.get("softcap", 0.0)), ptr(case.positions), ptr(case.slots), None))
        torch.cuda.synchronize()
        got[form] = out
    assert bool(torch.isfinite(got[0]).all())
    assert torch.equal(got[0], got[2])


def test_many_single_tokens_beside_portions_take_their_own_kernel(tmp_path):
    """bfloat16, 16 heads: 17 requests' single tokens are more than a workgroup a compute unit as tiles, so they go by themselves
    by the engine's own rule, from the step's first row on, with two portions behind them, and have the bits of tiles of 16
    rows; 16 of them go in the portions' tiles of 64 rows.  The portions are the same in all."""
    from celeg_amd.config import LayerSpec, ModelSpec, PartSpec, RunStep, register_architecture, registered_architectures
    from celeg_amd.engine import load_model
    from celeg_amd.weights.safetensors_io import write_safetensors
    if "SingleTokensAlone" not in registered_architectures():
        def build(cfg, shapes):
            W, rows = cfg["width"], cfg["rows"]
            block = LayerSpec(PartSpec.from_json(cfg["mixer"]), PartSpec("identity"), PartSpec("none"), PartSpec("identity"), "parallel")
            return ModelSpec("SingleTokensAlone", rows, W, 2048, PartSpec("embedding", {"vocab": rows, "width": W}, {"table": "table"}),
                             (block,), (RunStep(0, None, False),), PartSpec("identity"), PartSpec("hidden", {"width": W}))
        register_architecture("SingleTokensAlone", build)
    rows, W_, H, G, D = 256, 64, 16, 8, 32
    gen = torch.Generator().manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=gen)
    t = {"table": 1.5 * r(rows, W_), "q": 0.3 * r(H * D, W_), "k": 0.3 * r(G * D, W_), "v": 0.3 * r(G * D, W_), "o": 0.3 * r(W_, H * D)}
    part = {"kind": "biased_attention", "tensors": {n: n for n in "qkvo"},
            "params": {"width": W_, "heads": H, "kv_heads": G, "head_dim": D, "v_dim": D, "scale": D ** -0.5, "sink_one": True, "taps": 0}}
    with open(tmp_path / "config.json", "w") as fh:
        json.dump({"architectures": ["SingleTokensAlone"], "width": W_, "rows": rows, "mixer": part}, fh)
    write_safetensors(str(tmp_path / "model.safetensors"), {k: v.bfloat16().contiguous() for k, v in t.items()})
    tokens = torch.randint(0, rows, (19, 200), generator=gen).tolist()
    for singles in (17, 16):
        entry = lambda i, a, b: {"id": f"r{i}", "tokens": tokens[i][a:b], "want": list(range(b - a))}
        steps = [{"entries": [entry(i, 0, 40 + 7 * i)], "end": []} for i in range(singles)]
        steps.append({"entries": [entry(17, 0, 90)] + [entry(i, 40 + 7 * i, 41 + 7 * i) for i in range(singles)] + [entry(18, 0, 33)], "end": []})
        got = {}
        for form in (-1, 0, 1):
            lm = load_model(str(tmp_path), dtype="bfloat16", device=DEV, page_tokens=PAGE, n_pages=19 * 13, max_requests=19, max_context=200,
                            max_batched_tokens=256)
            lm.set_knob("biased_rows_form", form)
            got[form] = EngineDriver(lm).run(steps)
        for i in range(singles):
            assert torch.equal(got[-1][f"r{i}"][-1], got[0 if singles == 17 else 1][f"r{i}"][-1]), i
        for name in ("r17", "r18"):
            assert torch.equal(got[-1][name], got[1][name]), name


# (the last but one: 16 heads of 128, whose sums fill 64 KB of LDS)
@pytest.mark.parametrize("H,G,D,contexts,window,size,bias", [
    (16, 8, 64, [1100, 1, 32, 33], 1024, 1.0, 0.0), (16, 8, 64, [1500, 641, 1024, 700, 1100, 999, 640, 8], 1024, 4.0, -7.0),
    (4, 2, 96, [1500, 700, 701], 700, 2.0, -6.0), (16, 1, 128, [2000, 1999], 0, 1.0, -7.0), (4, 4, 32, [640, 513, 17], 0, 2.0, -6.0)])
def test_sigmoid_attention_of_single_tokens_is_no_further_from_the_exact_result(H, G, D, contexts, window, size, bias):
    """Over one, five and eight parts of the keys.  The weights' rounding to bfloat16 is most of the distance in both forms; the sums,
    32-bit in either order, move it by less than a hundredth."""
    case = Decoding(contexts, H, G, D, D, seed=D, spread=size)
    temp, beta = torch.linspace(0.7, 1.3, H, device=DEV), torch.full((H,), bias, device=DEV)
    want = torch.empty(case.n, H * D, dtype=torch.float64, device=DEV)
    for i, c in enumerate(contexts):
        k, v = case.keys_and_values(i)
        first = max(0, c - window) if window else 0
        k, v = (x[first:].repeat_interleave(H // G, 1) for x in (k, v))
        s = (k * case.q[i].double().view(1, H, D)).sum(-1) / math.sqrt(D) * temp.double() + beta.double()
        want[i] = (torch.sigmoid(s)[:, :, None] * v).sum(0).reshape(-1)
    lib, off = native.lib(), {}
    sums = torch.empty(case.n * H * D * 8, device=DEV)
    for parts in (0, 1, 5, 8):
        out = torch.full((case.n, H * D), float("nan"), dtype=BF, device=DEV)
        if parts:
            check(lib.celeg_sigmoid_attention_single(ptr(case.q), H * D, ptr(case.k), ptr(case.v), ptr(case.table), case.per, ptr(case.slots),
                                                     ptr(case.positions), ptr(temp), ptr(beta), None, 0, ptr(out), H * D, ptr(sums), parts, case.n,
                                                     H, G, D, PAGE, case.layers, case.layer, ctypes.c_float(1 / math.sqrt(D)), window, None))
        else:
            check(lib.celeg_sigmoid_attention_fast(0, ptr(case.q), H * D, ptr(case.k), ptr(case.v), ptr(case.table), case.per, ptr(case.cu),
                                                   ptr(case.slots), ptr(case.positions), case.n, case.n, ptr(temp), ptr(beta), None, 0, ptr(out),
                                                   H * D, H, G, D, PAGE, case.layers, case.layer, ctypes.c_float(1 / math.sqrt(D)), window, None))
        torch.cuda.synchronize()
        off[parts] = float((out.double() - want).norm() / want.norm())
    assert max(off[parts] for parts in (1, 5, 8)) <= 1.01 * off[0] <= 4e-3


@pytest.mark.parametrize("dtype", [torch.float32, BF])
@pytest.mark.parametrize("D,window", [(64, 0), (64, 24), (160, 96), (256, 65), (256, 128)])
def test_general_attention_of_few_rows_has_the_bits_of_many(dtype, D, window):
    """Heads of 64: few rows ask for a chunk of more than 16 keys as a whole, shorter ones and many rows for 16 at a time; heads beyond 128
    with windows of 65 to 128 keys: few rows have no condition round a key's product. The same bits, and 64 bits' results, with contexts
    at the edges and anything behind a request's last key."""
    contexts, H, G = [1, 2, 15, 16, 17, 18, 31, 32, 33, 64, 65, 79, 80, 81, 129, 300], 16, 8
    d = Decoding(contexts, H, G, D, D)
    q, k, v = d.q.to(dtype), d.k.to(dtype), d.v.to(dtype)
    times = 5                                     # 80 rows of 16 heads are more than what counts as few

    def run(n):
        # (all of them named: an address keeps no tensor alive)
        out, rows, slots, positions = torch.empty(n * d.n, H * D, dtype=dtype, device=DEV), q.repeat(n, 1), d.slots.repeat(n), d.positions.repeat(n)
        check(native.lib().celeg_paged_attention(
            ptr(rows), H * D, ptr(k), ptr(v), 0 if dtype == torch.float32 else 1, ptr(d.table), d.per, ptr(slots), ptr(positions), ptr(out),
            H * D, n * d.n, H, G, D, PAGE, d.layers, d.layer, ctypes.c_float(0.125), window, None))
        torch.cuda.synchronize()
        return out

    few = run(1)
    assert torch.equal(run(times), few.repeat(times, 1))
    for i, c in enumerate(contexts):
        keys, values = (t[-window:].cpu().repeat_interleave(H // G, 1) for t in d.keys_and_values(i))
        w = torch.softmax((d.q[i].double().cpu().view(H, D) * keys).sum(-1).T * 0.125, -1)
        want = (w.T[..., None] * values).sum(0).reshape(-1)
        # 32-bit scores, weights and sums of up to 300 keys, each step within 2^-24 of the magnitudes; a bfloat16 result is rounded
        bound = 2.0 ** -24 * 400 * float(values.abs().max()) + (0.0 if dtype == torch.float32 else 2.0 ** -8) * want.abs()
        assert bool(((few[i].double().cpu() - want).abs() <= bound).all()), c
