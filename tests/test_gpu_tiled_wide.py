"""Tiled products beyond one round of workgroups (the tile of 256x256 among those chosen), and which steps of streams wider
than 1,024 take the tiles."""
import pytest
import torch

from helpers import assert_close_bf16, random_tokens
from kernel_ops import HipOps

DEV = "cuda:0"
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    ops = HipOps()
    yield ops
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(-1)


def randn(*shape, seed, scale=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(dtype).to(DEV)


# the last: by the rule, two rounds of 256x256 (SwiGLU), and 256x192 (into the stream and stored)
@pytest.mark.gpu
@pytest.mark.parametrize("shape,M,N,K", [(11, 1, 4, 64), (11, 257, 132, 192), (11, 255, 256, 320), (11, 300, 516, 1088), (-1, 2047, 8192, 128)])
@pytest.mark.parametrize("epilogue", ["store", "residual", "swiglu"])
def test_square_tiles_give_the_bits_of_small_ones(ops, epilogue, shape, M, N, K):
    """Every element's products are added in the order of k, whatever the tile: the same bits as 32x64 gives."""
    a = randn(M, K, seed=51, dtype=BF)
    w = randn(N * (2 if epilogue == "swiglu" else 1), K, seed=52, scale=0.1, dtype=BF)
    results = []
    for force in (0, shape):
        ops._lib("gemm_tiles").celeg_gemm_tiles_force(force)
        if epilogue == "residual":
            out, copy = torch.ones(M + 1, N, device=DEV), torch.zeros(M, N, dtype=BF, device=DEV)
            ops.tiled_linear(a, w, out[:M], epilogue="residual", out_bf16=copy)
        else:
            out, copy = torch.ones(M + 1, N, dtype=BF, device=DEV), None
            stats = randn(M, 4, seed=53).abs() + 0.1
            ops.tiled_linear(a, w, out[:M], epilogue=epilogue, stats=stats, stat_blocks=4, eps=1e-5)
        results.append((out, copy))
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(-1)
    assert torch.equal(results[0][0], results[1][0]) and bool((results[1][0][M] == 1).all())
    assert results[0][1] is None or torch.equal(results[0][1], results[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("width,rows,tiles", [(1088, 70, True), (1536, 1100, True), (1600, 65, True), (1600, 1024, True), (1600, 1025, False),
                                              (1600, 1599, False), (1600, 1600, True), (2112, 256, True), (2112, 257, False), (2624, 65, False)])
def test_which_steps_of_wide_streams_take_the_tiles(tmp_path, width, rows, tiles):
    """By the step's rows, where nobody has chosen, and never where the library was chosen; the logits against 64 bits."""
    import plain_lfm2 as plain
    from celeg_amd.engine import Engine
    from celeg_amd.sampling import GREEDY
    from celeg_amd.weights import write_random_model
    config = {"architectures": ["Lfm2ForCausalLM"], "vocab_size": 512, "hidden_size": width, "num_hidden_layers": 2,
              "layer_types": ["conv", "full_attention"], "num_attention_heads": width // 64, "num_key_value_heads": 1, "head_dim": 64,
              "intermediate_size": 1024, "block_auto_adjust_ff_dim": False, "rope_theta": 10000.0, "conv_L_cache": 3, "conv_bias": False,
              "tie_word_embeddings": True, "norm_eps": 1e-5, "max_position_embeddings": 2048, "eos_token_id": 7}
    folder = write_random_model(config, str(tmp_path), seed=3, dtype=BF, std=0.03)
    cfg, W = plain.load_model_folder(folder)
    prompt = random_tokens(512, rows, seed=rows)
    want = plain.model_logits(cfg, W, prompt)[-1:]
    for backend in ("auto", "library"):
        engine = Engine.from_folder(folder, dtype="bfloat16", device=DEV, max_active_requests=1, n_pages=rows // 16 + 2,
                                    max_batched_tokens=2048, prefill_chunk_tokens=2048, gemm_backend=backend)
        engine.generate([prompt], max_new_tokens=1, generation=GREEDY, eos_token_ids=[])
        assert_close_bf16(engine.last_logits, want, backend)
        paths = engine.loaded.paths()
        assert (paths["tiled"] > 0) == (paths["tiled_qkv"] > 0) == (tiles and backend == "auto"), paths
        engine.close()
