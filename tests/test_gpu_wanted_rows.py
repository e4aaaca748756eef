"""The last layer's feed-forward for the wanted rows of a step alone: the logits against the plain implementation and against
the pass over all rows, and the kernel that takes the rows out."""
import ctypes

import pytest
import torch

import plain_lfm2 as plain
from helpers import assert_close, random_tokens
from kernel_ops import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,n,width,inner,side", [(70, 1, 64, 64, False), (70, 33, 64, 192, True), (9, 4, 1024, 4608, True), (65, 65, 6, 10, False),
                                                  (3, 5, 2052, 8, False), (300, 64, 1028, 2056, True)])
def test_rows_taken_out(dtype, T, n, width, inner, side):
    lib = HipOps()._lib("layer_glue")
    gen = torch.Generator().manual_seed(T * n)
    h = torch.randn(T, width, generator=gen).to(DEV)
    a = torch.randn(T, inner + 8, generator=gen).to(dtype).to(DEV)[:, :inner]       # (rows of a wider matrix)
    rows = torch.randint(0, T, (n,), generator=gen, dtype=torch.int32).to(DEV)
    h_out = torch.full((n + 1, width), 7.0, device=DEV)
    a_out = torch.full((inner // 8, n + 1, 8) if side else (n + 1, inner), 7.0, dtype=dtype, device=DEV)
    ld, k8 = (8, (n + 1) * 8) if side else (inner, 8)
    p, ll = ctypes.c_void_p, ctypes.c_longlong
    rc = lib.celeg_gather_rows(p(rows.data_ptr()), n, p(h.data_ptr()), p(h_out.data_ptr()), width, p(a.data_ptr()), ll(inner + 8),
                               p(a_out.data_ptr()), ll(ld), ll(k8), inner, 0 if dtype == torch.float32 else 1,
                               p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    got = a_out.permute(1, 0, 2).reshape(n + 1, inner) if side else a_out
    assert torch.equal(h_out[:n], h[rows.long()]) and bool((h_out[n] == 7).all())
    assert torch.equal(got[:n], a[rows.long()]) and bool((got[n] == 7).all())


# entries (tokens, wanted places from the end) of the steps of one run: portions without wanted rows, single tokens beside
# prompts, several places of one entry, and (65 rows, 33 wanted) a step that keeps all rows
STEPS = [[(0, 70, [])], [(0, 66, [1]), (1, 40, [1, 2, 40])], [(2, 129, [129, 1]), (0, 1, [1]), (1, 1, [1])], [(3, 65, list(range(1, 34)))],
         [(3, 160, list(range(1, 77)))]]


@pytest.mark.parametrize("dtype,last,width,backend", [("bfloat16", "conv", 128, "auto"), ("bfloat16", "full_attention", 128, "auto"),
                                                      ("bfloat16", "conv", 128, "library"), ("float32", "full_attention", 128, "auto"),
                                                      ("float32", "conv", 192, "auto")])
def test_logits_of_the_wanted_rows(tmp_path, dtype, last, width, backend):
    from celeg_amd.engine import StepEntry, load_model
    from celeg_amd.weights import write_random_model
    config = {"architectures": ["Lfm2ForCausalLM"], "vocab_size": 320, "hidden_size": width, "num_hidden_layers": 3,
              "layer_types": ["conv", "full_attention", last], "num_attention_heads": width // 64, "num_key_value_heads": 1, "head_dim": 64,
              "intermediate_size": 448, "block_auto_adjust_ff_dim": False, "rope_theta": 10000.0, "conv_L_cache": 3, "conv_bias": False,
              "tie_word_embeddings": True, "norm_eps": 1e-5, "max_position_embeddings": 512, "eos_token_id": 7}
    folder = write_random_model(config, str(tmp_path), seed=5, dtype=getattr(torch, dtype), std=0.05)
    cfg, W = plain.load_model_folder(folder)
    results = []
    for only in (0, 1):
        lm = load_model(folder, dtype=dtype, page_tokens=16, n_pages=80, max_requests=4, max_batched_tokens=512, gemm_backend=backend)
        lm.set_knob("wanted_rows_only", only)
        slots, tokens, seen = {}, {i: random_tokens(320, 400, seed=60 + i) for i in range(4)}, {}
        for step in STEPS:
            entries, want = [], []
            for request, n, from_end in step:
                slot = slots.setdefault(request, lm.cache.open() if request not in slots else None)
                pos = seen.get(request, 0)
                assert lm.cache.prepare(slot, pos, n)
                entries.append(StepEntry(slot, pos, tokens[request][pos:pos + n], [n - k for k in from_end]))
                want += [(request, pos + n - k) for k in from_end]
                seen[request] = pos + n
            got = lm.runner.step(entries)
            assert got.shape[0] == len(want)
            results.append((only, got.clone(), want))
        lm.close()
    whole = {r: plain.model_logits(cfg, W, tokens[r]) for r in range(4)}
    for only, got, want in results:
        if not want:
            continue
        ref = torch.stack([whole[r][at] for r, at in want])
        assert_close(got, ref, dtype, f"{dtype}/{last}/{backend}/wanted only {only}")


def one_prompt(folder, wanted, T=150, backend="auto"):
    """One step of a prompt of T tokens with its last `wanted` rows wanted: their logits and what each kernel family launched."""
    from celeg_amd.engine import StepEntry, load_model
    lm = load_model(folder, dtype="bfloat16", page_tokens=16, n_pages=40, max_requests=4, max_batched_tokens=512, gemm_backend=backend)
    tokens = random_tokens(320, T, seed=wanted)
    slot = lm.cache.open()
    assert lm.cache.prepare(slot, 0, T)
    before = lm.knobs()["paths"]
    got = lm.runner.step([StepEntry(slot, 0, tokens, list(range(T - wanted, T)))]).clone()
    after = lm.knobs()["paths"]
    lm.close()
    return got.double().cpu(), tokens, {k: after[k] - before[k] for k in after}


def small_config(width, vocab=320, tied=True, ff=448):
    return {"architectures": ["Lfm2ForCausalLM"], "vocab_size": vocab, "hidden_size": width, "num_hidden_layers": 2,
            "layer_types": ["conv", "full_attention"], "num_attention_heads": max(1, width // 64), "num_key_value_heads": 1, "head_dim": 64,
            "intermediate_size": ff, "block_auto_adjust_ff_dim": False, "rope_theta": 10000.0, "conv_L_cache": 3, "conv_bias": False,
            "tie_word_embeddings": tied, "norm_eps": 1e-5, "max_position_embeddings": 512, "eos_token_id": 7}


# (8 and fewer, 9 to 64 and more rows have kernels of their own; 16,400 columns are more than those of up to 16 rows fold a norm into)
@pytest.mark.parametrize("wanted", [1, 8, 9, 16, 33, 64, 75])
@pytest.mark.parametrize("vocab", [320, 16400])
def test_the_head_reads_the_output_table_as_it_is(tmp_path, wanted, vocab):
    """Every entry of the table is 1.5 times a power of two and every weight of the final norm 1 + 2^-7: their product lies half way
    between two bfloat16 numbers and rounds to 1.515625 of that power, 2^-8.6 too much.  Logits from the table as it is have no
    such bias: what the roundings of the layers leave of one, 2^-8 a value over 128 values of a row and more, is a tenth of it."""
    from celeg_amd.weights import write_random_model, write_safetensors
    config = small_config(128, vocab, tied=False)
    folder = write_random_model(config, str(tmp_path), seed=3, dtype=torch.bfloat16, std=0.05)
    cfg, W = plain.load_model_folder(folder)
    gen = torch.Generator().manual_seed(4)
    signs = torch.randint(0, 2, W["lm_head.weight"].shape, generator=gen) * 2.0 - 1.0
    W["lm_head.weight"] = (signs * 1.5 * 2.0 ** -torch.randint(3, 6, signs.shape, generator=gen)).double()
    W["model.embedding_norm.weight"] = torch.full_like(W["model.embedding_norm.weight"], 1 + 2.0 ** -7)
    write_safetensors(f"{folder}/model.safetensors", {k: v.to(torch.bfloat16) for k, v in W.items()}, metadata={"format": "pt"})
    got, tokens, _ = one_prompt(folder, wanted)
    ref = plain.model_logits(cfg, W, tokens)[-wanted:]
    assert got.shape == ref.shape
    bias = float((got * ref).sum() / (ref * ref).sum()) - 1
    assert abs(bias) < 1e-3, bias


# (480: the products of many rows want a multiple of 64, those of few rows one of 32; a single layer, whose mixer takes the norm along)
@pytest.mark.parametrize("width,ff,backend", [(128, 448, "library"), (1152, 448, "auto"), (128, 480, "auto")])
@pytest.mark.parametrize("wanted", [1, 8, 9, 33, 64])
def test_no_norm_is_folded_where_the_whole_step_folds_none(tmp_path, width, ff, backend, wanted):
    """Feed-forwards of many rows that the library's products make read every weight as it is stored; so do the rows that are left
    of such a step.  (Of the fused products the one into the stream behind the mixer, which has no norm, remains.)"""
    from celeg_amd.weights import write_random_model
    config = small_config(width, ff=ff)
    if ff == 480:
        config.update(num_hidden_layers=1, layer_types=["full_attention"])
    folder = write_random_model(config, str(tmp_path), seed=5, dtype=torch.bfloat16, std=0.05 if width < 1000 else 0.03)
    got, tokens, paths = one_prompt(folder, wanted, backend=backend)
    cfg, W = plain.load_model_folder(folder)
    assert_close(got, plain.model_logits(cfg, W, tokens)[-wanted:], "bfloat16", f"{width}/{ff}/{backend}/{wanted}")
    assert paths["linear_few_rows"] > 0
    assert paths["fused_rows"] + paths["fused_sliced"] <= (1 if ff == 480 else 0), paths


@pytest.mark.parametrize("dtype,last", [("bfloat16", "conv"), ("bfloat16", "full_attention"), ("float32", "full_attention")])
@pytest.mark.parametrize("wanted", [9, 16, 17, 33, 64, 65])
def test_logits_of_9_to_64_wanted_rows(tmp_path, dtype, last, wanted):
    """As ragged prompts and a server have them: one row of each of so many prompts of 2 to 5 tokens, and a step behind."""
    from celeg_amd.engine import StepEntry, load_model
    from celeg_amd.weights import write_random_model
    config = small_config(128)
    config["layer_types"] = ["full_attention", last]
    folder = write_random_model(config, str(tmp_path), seed=6, dtype=getattr(torch, dtype), std=0.05)
    cfg, W = plain.load_model_folder(folder)
    lm = load_model(folder, dtype=dtype, page_tokens=16, n_pages=80, max_requests=72, max_batched_tokens=512)
    tokens = [random_tokens(320, 2 + i % 4 + 2 + (70 if i == 0 else 0), seed=80 + i) for i in range(wanted)]
    slots, seen = [lm.cache.open() for _ in tokens], [0] * wanted
    for n in ([len(t) - 2 for t in tokens], [1] * wanted):
        entries = []
        for i, slot in enumerate(slots):
            assert lm.cache.prepare(slot, seen[i], n[i])
            entries.append(StepEntry(slot, seen[i], tokens[i][seen[i]:seen[i] + n[i]], [n[i] - 1]))
            seen[i] += n[i]
        got = lm.runner.step(entries)
        assert_close(got, torch.stack([plain.model_logits(cfg, W, t[:s])[-1] for t, s in zip(tokens, seen)]), dtype, f"{dtype}/{last}/{wanted}")
    lm.close()


@pytest.mark.parametrize("dtype,last,backend", [("bfloat16", "conv", "auto"), ("bfloat16", "full_attention", "auto"),
                                                ("bfloat16", "conv", "library"), ("float32", "conv", "auto")])
def test_recorded_steps_stay_good_however_many_rows_are_wanted(tmp_path, dtype, last, backend):
    """Twelve requests decoded together between steps of 200 rows: the first of these makes every buffer of the others."""
    from celeg_amd.engine import StepEntry, load_model
    from celeg_amd.weights import write_random_model
    config = small_config(128)
    config["layer_types"] = ["full_attention", last]
    folder = write_random_model(config, str(tmp_path), seed=8, dtype=getattr(torch, dtype), std=0.05)
    lm = load_model(folder, dtype=dtype, page_tokens=16, n_pages=400, max_requests=12, max_batched_tokens=256, gemm_backend=backend)
    slots, seen = [lm.cache.open() for _ in range(12)], [0] * 12

    def step(*entries):
        batch = []
        for i, n, wanted in entries:
            assert lm.cache.prepare(slots[i], seen[i], n)
            batch.append(StepEntry(slots[i], seen[i], random_tokens(320, n, seed=seen[i]), list(range(n - wanted, n))))
            seen[i] += n
        lm.runner.step(batch)
        return lm.runner.counters()["captures"]
    singles = [(i, 1, 1) for i in range(12)]
    step((0, 120, 60), (1, 80, 40))
    step(*singles)
    recorded = step(*singles)
    for wanted in (1, 9, 33, 70, 100):
        step((2 + wanted % 5, 50, wanted // 2), (8, 150, wanted - wanted // 2))
        assert step(*singles) == recorded, wanted
        seen[8] = 0
    lm.close()


@pytest.mark.parametrize("arrangement", ["pre_norm", "sandwich_norm"])
@pytest.mark.parametrize("shared", [False, True])
def test_a_feed_forward_that_reads_the_step_is_given_all_of_it(tmp_path, arrangement, shared):
    """A feed-forward from outside goes by its rows' tokens, places and requests, as the last layer's and as what routed experts
    share: it is given every row and the step's arrays, however few rows are wanted."""
    from celeg_amd.config import LayerSpec, ModelSpec, PartSpec, RunStep, register_architecture, registered_architectures
    from celeg_amd.engine import StepEntry, load_model
    from celeg_amd.parts import as_tensor, int_array, on_stream, register_part, registered_parts
    from celeg_amd.weights import write_random_model

    class ByToken:
        def __init__(self, spec):
            pass

        def describe(self):
            return {"graph_safe": False}

        def forward(self, args):
            step, rows = args.step, int(args.x.shape[0])
            if rows != step.n_tokens or not (step.token_ids and step.positions and step.host_seq_start and step.host_cu_seqlens) or \
                    step.host_cu_seqlens[step.n_seqs] != rows:
                raise RuntimeError("the step is not whole")
            with on_stream(args):
                by = int_array(step.token_ids, rows).float() + 0.5 * int_array(step.positions, rows).float()
                as_tensor(args.out).copy_(as_tensor(args.x) * (0.01 * by)[:, None])

    if "by_token" not in registered_parts("ffn"):
        register_part("ffn", "by_token", ByToken)

    def build(cfg, shapes):
        H, V = cfg["width"], cfg["vocab"]
        norm = lambda name: PartSpec("rmsnorm", {"width": H, "eps": 1e-5}, {"weight": name})
        ffn = PartSpec("by_token")
        if cfg["shared"]:
            names = {"router": "router"}
            for e in range(2):
                names.update({f"gate.{e}": f"{e}.g", f"up.{e}": f"{e}.u", f"down.{e}": f"{e}.d"})
            ffn = PartSpec("routed_experts", {"width": H, "ff": 32, "experts": 2, "top": 1, "shared": ffn}, names)
        layer = LayerSpec(PartSpec("none", {"width": H}), norm("n1"), ffn, norm("n2"), cfg["arrangement"],
                          **({"mixer_post_norm": norm("n3"), "ffn_post_norm": norm("n4")} if cfg["arrangement"] == "sandwich_norm" else {}))
        return ModelSpec("ByToken", V, H, 256, PartSpec("embedding", {"vocab": V, "width": H}, {"table": "emb"}), (layer,), (RunStep(0),),
                         norm("final"), PartSpec("hidden", {"width": H}))

    if "ByToken" not in registered_architectures():
        register_architecture("ByToken", build)
    config = {"architectures": ["ByToken"], "width": 32, "vocab": 90, "shared": shared, "arrangement": arrangement}
    folder = write_random_model(config, str(tmp_path), seed=7, dtype=torch.float32, std=0.3)
    lm = load_model(folder, dtype="float32", page_tokens=16, n_pages=40, max_requests=4, max_batched_tokens=256)
    tokens = random_tokens(90, 80, seed=3)

    def step(wanted):
        slot = lm.cache.open()
        assert lm.cache.prepare(slot, 0, 80)
        got = lm.runner.step([StepEntry(slot, 0, tokens, wanted)]).clone()
        lm.cache.close(slot)
        return got
    whole = step(list(range(80)))
    for wanted in ([79], [3, 70, 79], []):
        assert torch.equal(step(wanted), whole[wanted])
    lm.close()
