"""How often single tokens' steps are recorded: once for every bound on the context at which their launches change."""
import pytest
import torch

from helpers import random_tokens

pytestmark = pytest.mark.gpu


def recordings(lm, requests, contexts):
    """Recordings made behind the one for contexts[0], after a step of `requests` single tokens at each of these contexts.  (Nobody
    reads what the pages hold ahead of the tokens.  The first step brings so many pages that their list gets a buffer of its own,
    behind which it is recorded once more.)"""
    from celeg_amd.engine import StepEntry
    slots = [lm.cache.open() for _ in range(requests)]
    for slot in slots:
        assert lm.cache.prepare(slot, 0, max(contexts))
    seen = []
    for context in [contexts[0]] + contexts:
        lm.runner.step([StepEntry(slot, context - 1, random_tokens(60, 1, seed=slot), [0]) for slot in slots])
        seen.append(lm.runner.counters()["captures"])
    return [n - seen[1] for n in seen[1:]]


# pairs of request and key/value head: 8 and 56 (one workgroup each up to 640 keys), 64 (1,024), 96 and 128 (4,096); and 128
# requests, whose attention prepares the new keys itself up to 2,048 keys
@pytest.mark.parametrize("requests,kv_heads,after", [(1, 8, [0, 0, 1, 1, 1]), (8, 7, [0, 0, 1, 1, 1]), (8, 8, [0, 0, 0, 1, 1]),
                                                     (16, 6, [0, 0, 0, 0, 0]), (16, 8, [0, 0, 0, 0, 0]), (128, 1, [0, 0, 0, 1, 1])])
def test_softmax_attention(tmp_path, requests, kv_heads, after):
    from celeg_amd.engine import load_model
    from celeg_amd.weights import write_random_model
    config = {"architectures": ["Lfm2ForCausalLM"], "vocab_size": 60, "hidden_size": 64 * kv_heads, "num_hidden_layers": 1, "layer_types": ["full_attention"],
              "num_attention_heads": kv_heads, "num_key_value_heads": kv_heads, "head_dim": 64, "intermediate_size": 64,
              "block_auto_adjust_ff_dim": False, "rope_theta": 10000.0, "conv_L_cache": 3, "conv_bias": False, "tie_word_embeddings": True,
              "norm_eps": 1e-5, "max_position_embeddings": 2048, "eos_token_id": 7}
    folder = write_random_model(config, str(tmp_path), seed=2, dtype=torch.bfloat16, std=0.05)
    lm = load_model(folder, dtype="bfloat16", page_tokens=16, n_pages=requests * 66 + 2, max_requests=requests, max_batched_tokens=256)
    assert recordings(lm, requests, [600, 640, 641, 1030, 600]) == after
    lm.close()


def test_two_kinds_of_attention(tmp_path):
    """Sigmoid attention is cut into parts beyond 640 keys, softmax attention of 64 pairs beyond 1,024: steps of a model with both are
    recorded for each."""
    from celeg_amd.config import LayerSpec, ModelSpec, PartSpec, RunStep, register_architecture, registered_architectures
    from celeg_amd.engine import load_model
    from celeg_amd.weights import write_random_model

    def build_spec(cfg, shapes):
        width = cfg["width"]
        norm = lambda name: PartSpec("rmsnorm", {"width": width, "eps": 1e-5}, {"weight": name})
        rope = PartSpec("rope", {"theta": 100.0, "head_dim": 64})
        sizes = {"width": width, "heads": 8, "kv_heads": 8, "head_dim": 64, "qk_norm": False}
        layers = []
        for i, mixer in enumerate((PartSpec("gqa_attention", dict(sizes, position=rope),
                                            {"q_proj": "0.q", "k_proj": "0.k", "v_proj": "0.v", "out_proj": "0.o"}),
                                   PartSpec("sigmoid_attention", dict(sizes, position=rope), {"q": "1.q", "k": "1.k", "v": "1.v", "o": "1.o"}))):
            ffn = PartSpec("swiglu", {"width": width, "ff": 64}, {"gate": f"{i}.g", "up": f"{i}.u", "down": f"{i}.d"})
            layers.append(LayerSpec(mixer, norm(f"{i}.n1"), ffn, norm(f"{i}.n2")))
        return ModelSpec("BothAttentions", cfg["vocab"], width, 2048, PartSpec("embedding", {"vocab": cfg["vocab"], "width": width}, {"table": "emb"}),
                         tuple(layers), tuple(RunStep(i) for i in range(len(layers))), norm("final"),
                         PartSpec("tied_head", {"vocab": cfg["vocab"], "width": width}))

    if "BothAttentions" not in registered_architectures():
        register_architecture("BothAttentions", build_spec)
    folder = write_random_model({"architectures": ["BothAttentions"], "width": 64, "vocab": 60}, str(tmp_path), seed=2, dtype=torch.bfloat16,
                                std=0.05)
    lm = load_model(folder, dtype="bfloat16", page_tokens=16, n_pages=8 * 66 + 2, max_requests=8, max_batched_tokens=256)
    assert recordings(lm, 8, [600, 640, 641, 1024, 1030]) == [0, 0, 1, 1, 2]
    lm.close()


def test_room_for_parts_is_what_parts_need(tmp_path):
    """1,024 requests of 16 heads take their pairs whole at any context: no room for parts, of which 64 a head would be 277 MB.  (The
    rest of a step of so many rows, recorded, is 124 MB.)"""
    from celeg_amd.engine import load_model
    from celeg_amd.weights import write_random_model
    config = {"architectures": ["Lfm2ForCausalLM"], "vocab_size": 60, "hidden_size": 1024, "num_hidden_layers": 1, "layer_types": ["full_attention"],
              "num_attention_heads": 16, "num_key_value_heads": 8, "head_dim": 64, "intermediate_size": 64,
              "block_auto_adjust_ff_dim": False, "rope_theta": 10000.0, "conv_L_cache": 3, "conv_bias": False, "tie_word_embeddings": True,
              "norm_eps": 1e-5, "max_position_embeddings": 4096, "eos_token_id": 7}
    folder = write_random_model(config, str(tmp_path), seed=2, dtype=torch.bfloat16, std=0.05)
    lm = load_model(folder, dtype="bfloat16", page_tokens=16, n_pages=4200, max_requests=1024, max_batched_tokens=1024)
    recordings(lm, 1, [40])          # (the kernels' code and what a step of one request needs)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    recordings(lm, 1000, [40])
    torch.cuda.synchronize()
    taken = before - torch.cuda.mem_get_info()[0]
    lm.close()
    assert taken < 200 << 20, taken
