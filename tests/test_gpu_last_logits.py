"""The last step's logits on the host: their sizes alone, all of them, and the first of them."""
import ctypes

import numpy as np
import pytest
import torch

import plain_lfm2 as plain
from helpers import WEIGHT_STD, assert_close_f32, random_tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("requests", [1, 3])
def test_sizes_whole_and_parts(model_folders, requests):
    from celeg_amd import native
    from celeg_amd.engine import Engine
    from celeg_amd.sampling import GREEDY
    folder = model_folders("B", torch.float32, WEIGHT_STD)
    cfg, W = plain.load_model_folder(folder)
    V = cfg["vocab_size"]
    engine = Engine.from_folder(folder, dtype="float32", max_active_requests=4, n_pages=40, max_batched_tokens=64)
    call = native.lib().celeg_engine_last_logits
    rows, vocab = ctypes.c_int32(-1), ctypes.c_int32(-1)
    native.check(call(engine.native.handle, None, 0, ctypes.byref(rows), ctypes.byref(vocab)))
    assert (rows.value, vocab.value) == (0, 0) and tuple(engine.last_logits.shape) == (0, 0)       # before any step
    prompts = [random_tokens(V, n, seed=40 + n) for n in (5, 9, 14)[:requests]]
    engine.generate(prompts, max_new_tokens=1, generation=GREEDY, eos_token_ids=[])
    native.check(call(engine.native.handle, None, 0, ctypes.byref(rows), ctypes.byref(vocab)))
    assert (rows.value, vocab.value) == (requests, V)
    whole = engine.last_logits
    assert_close_f32(whole, torch.stack([plain.model_logits(cfg, W, p)[-1] for p in prompts]))
    for capacity in (0, 1, V - 1, V, V + 1, requests * V, requests * V + 7):
        out = np.full(requests * V + 8, 7.0, dtype=np.float32)
        native.check(call(engine.native.handle, out.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), capacity, None, None))
        n = min(capacity, requests * V)
        assert np.array_equal(out[:n], whole.numpy().reshape(-1)[:n]) and (out[n:] == 7.0).all()
