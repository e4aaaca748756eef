"""The short convolution over the rows of a step of 9 to 64, inside the product ahead of it: requests that begin, go on and end
anywhere among the rows, fewer rows than taps, single tokens beside portions, states carried from step to step."""
import pytest
import torch

import plain_lfm2 as plain
from helpers import assert_close_bf16, random_tokens

pytestmark = pytest.mark.gpu

# (request, tokens) of each step: 9 rows (a tile of 16), 16 and 17, 32 and 33, 63 and 64 (the largest), requests of 1, 2 and 3 rows,
# steps of 8 and 65 rows between them (other kernels read and write the same states)
STEPS = [[(0, 9)], [(1, 2), (0, 14)], [(2, 1), (1, 1), (0, 15)], [(2, 1), (3, 31)], [(3, 2), (2, 30), (1, 1)], [(0, 4), (1, 4)],
         [(3, 62), (2, 1)], [(0, 1), (1, 3), (2, 2), (3, 58)], [(0, 65)], [(0, 10), (1, 33), (3, 1), (2, 2)]]


@pytest.mark.parametrize("width,taps,bias", [(128, 3, False), (192, 2, True), (1152, 4, False), (2304, 3, True), (64, 9, False),
                                             (512, 9, False), (544, 2, True)])
def test_conv_rows(tmp_path, width, taps, bias):
    from celeg_amd.engine import StepEntry, load_model
    from celeg_amd.weights import write_random_model
    config = {"architectures": ["Lfm2ForCausalLM"], "vocab_size": 320, "hidden_size": width, "num_hidden_layers": 3,
              "layer_types": ["conv", "full_attention", "conv"], "num_attention_heads": max(2, width // 64), "num_key_value_heads": 1,
              "head_dim": 64, "intermediate_size": 448, "block_auto_adjust_ff_dim": False, "rope_theta": 10000.0, "conv_L_cache": taps,
              "conv_bias": bias, "tie_word_embeddings": True, "norm_eps": 1e-5, "max_position_embeddings": 512, "eos_token_id": 7}
    if width < 128:
        config.update(num_attention_heads=1)
    folder = write_random_model(config, str(tmp_path), seed=9, dtype=torch.bfloat16, std=0.05 if width < 1000 else 0.03)
    cfg, W = plain.load_model_folder(folder)
    tokens = {r: random_tokens(320, 256, seed=70 + r) for r in range(4)}
    runs = []
    for use in (0, 1):
        lm = load_model(folder, dtype="bfloat16", page_tokens=16, n_pages=80, max_requests=4, max_batched_tokens=128)
        lm.set_knob("use_conv_rows", use)
        slots, seen, out = [lm.cache.open() for _ in range(4)], [0] * 4, []
        for step in STEPS:
            entries = []
            for request, n in step:
                assert lm.cache.prepare(slots[request], seen[request], n)
                entries.append(StepEntry(slots[request], seen[request], tokens[request][seen[request]:seen[request] + n], [n - 1]))
                seen[request] += n
            out.append((lm.runner.step(entries).clone(), [(r, seen[r] - 1) for r, _ in step]))
        runs.append(out)
        lm.close()
    for (apart, want), (inside, _) in zip(*runs):
        assert_close_bf16(inside, torch.stack([plain.model_logits(cfg, W, tokens[r][:at + 1])[-1] for r, at in want]))
        if width <= 192:       # (K is cut alike and a row has few partial sums of squares: the same bits)
            assert torch.equal(apart, inside)


def test_where_the_convolution_is_inside():
    """Up to 16 rows from a width of 128 on, up to 32 from 512 and up to 64 from 2,048; elsewhere it is slower there."""
    from kernel_ops import HipOps
    ops = HipOps()
    for width, most in ((64, 0), (96, 0), (128, 16), (480, 16), (512, 32), (1024, 32), (2016, 32), (2048, 64), (4096, 64)):
        for rows in (1, 8, 9, 16, 17, 32, 33, 64, 65):
            assert ops.conv_rows_pay(rows, width) == (9 <= rows <= most), (rows, width)
