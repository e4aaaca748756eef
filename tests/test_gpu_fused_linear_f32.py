"""The 32-bit products of few rows with what surrounds them, called as the host code calls them: every epilogue at row counts on both
sides of a change of layout, columns and inner sizes beside a tile's, against 64 bits; and a model's logits with and without them."""
import ctypes

import pytest
import torch

import plain_lfm2 as plain
from celeg_amd import native
from helpers import random_tokens
from test_gpu_single_tokens import check, ptr

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 2.0 ** -24
STORE, RESIDUAL, SWIGLU, CONV = 0, 2, 3, 4


def call(x, w, y, N, epi, norm=None, bias=None, conv=None):
    taps, conv_b, state, slots = conv or (None, None, None, None)
    return native.lib().celeg_gemm_f32_fused(
        ptr(x), x.stride(0), ptr(w), w.stride(0), ptr(bias), ptr(y), y.stride(0), x.shape[0], N, x.shape[1], epi, ptr(norm),
        ctypes.c_float(1e-5), ptr(taps), ptr(conv_b), ptr(state), ctypes.c_size_t(0 if state is None else state.stride(0)), ptr(slots),
        0 if taps is None else taps.shape[1], None)


@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(1, 4), (5, 132), (33, 128), (20, 1000), (66, 2048), (1024, 1024)])
def test_every_epilogue_against_64_bits(M, N, K):
    gen = torch.Generator().manual_seed(M * 1000 + N + K)
    r = lambda *s: torch.randn(*s, generator=gen)
    x, norm = (2.0 * r(M, K)).to(DEV), (1.0 + 0.3 * r(K)).to(DEV)
    xd, nd = x.double(), norm.double()
    normed = xd / torch.sqrt((xd * xd).mean(-1, keepdim=True) + 1e-5) * nd

    def product(rows, w):
        """64-bit sums and a bound on 32-bit ones: 128 products a segment one after the other, 16 segments, the row's scale"""
        return rows @ w.double().T, (128 + 16 + 24) * EPS * (rows.abs() @ w.double().abs().T)

    # stored behind a norm
    w, b = (0.1 * r(N, K)).to(DEV), r(N).to(DEV)
    y = torch.full((M, N + 3), 7.0, device=DEV)[:, :N]
    check(call(x, w, y, N, STORE, norm, b))
    want, bound = product(normed, w)
    want = want + b.double()
    assert ((y.double() - want).abs() <= bound + EPS * want.abs() + 1e-30).all()
    # into the stream: the plain product's own sum, added in 32-bit
    h = r(M, N).to(DEV)
    plain_out, got = torch.empty(M, N, device=DEV), h.clone()
    check(native.lib().celeg_gemm_f32(ptr(x), K, ptr(w), K, ptr(b), ptr(plain_out), N, M, N, K, None))
    check(call(x, w, got, N, RESIDUAL, None, b))
    assert torch.equal(got, h + plain_out)
    # SwiGLU
    w2 = (0.1 * r(2 * N, K)).to(DEV)
    y = torch.empty(M, N, device=DEV)
    check(call(x, w2, y, N, SWIGLU, norm))
    g, eg = product(normed, w2[:N])
    u, eu = product(normed, w2[N:])
    silu = g * torch.sigmoid(g)
    assert ((y.double() - silu * u).abs() <= 1.1 * eg * u.abs() + 2 * silu.abs() * eu + 2 * eg * eu + 16 * EPS * (silu * u).abs() + 1e-30).all()
    # the short convolution, one new token per request, with its state
    for L in (1, 3, 8):
        w3, taps, cb = (0.1 * r(3 * N, K)).to(DEV), r(N, L).to(DEV), r(N).to(DEV)
        state = r(M + 2, 2, L, N).to(DEV)[:, 1]
        before, slots = state.clone(), torch.tensor([(3 * i + 1) % (M + 2) if (M + 2) % 3 else (i + 1) % (M + 2) for i in range(M)], dtype=torch.int32, device=DEV)
        check(call(x, w3, y, N, CONV, norm, None, (taps, cb, state, slots)))
        (B, eB), (C, eC), (X, eX) = (product(normed, w3[i * N:(i + 1) * N]) for i in range(3))
        old = before[slots.long()].double()
        bx, ebx = B * X, eB * X.abs() + B.abs() * eX + eB * eX + EPS * (B * X).abs()
        terms = torch.cat([old[:, 1:], bx[:, None]], 1) * taps.double().T[None]
        conv = terms.sum(1) + cb.double()
        econv = taps.double().T[-1].abs() * ebx + (L + 2) * EPS * (terms.abs().sum(1) + cb.double().abs())
        assert ((y.double() - C * conv).abs() <= eC * conv.abs() + C.abs() * econv + eC * econv + 2 * EPS * (C * conv).abs() + 1e-30).all()
        now = state[slots.long()]
        assert torch.equal(now[:, :L - 1], before[slots.long()][:, 1:])
        assert ((now[:, L - 1].double() - bx).abs() <= ebx).all()
        others = [s for s in range(M + 2) if s not in slots.tolist()]
        assert torch.equal(state[others], before[others])


@pytest.mark.parametrize("K", [2304, 4608])
def test_long_rows_go_into_the_stream_and_are_refused_behind_a_norm(K):
    gen = torch.Generator().manual_seed(K)
    for M in (1, 4, 5, 16):
        x, w, h = (torch.randn(*s, generator=gen).to(DEV) for s in ((M, K), (40, K), (M, 40)))
        plain_out, got = torch.empty(M, 40, device=DEV), h.clone()
        check(native.lib().celeg_gemm_f32(ptr(x), K, ptr(w), K, None, ptr(plain_out), 40, M, 40, K, None))
        check(call(x, w, got, 40, RESIDUAL))
        assert torch.equal(got, h + plain_out)
        assert call(x, w, got, 40, STORE, torch.ones(K, device=DEV)) != 0


@pytest.mark.parametrize("M", [1, 3, 8, 9, 16])
@pytest.mark.parametrize("K", [256, 260, 380, 384, 388, 516, 640, 768, 896, 1000, 1020, 1024])
def test_the_norm_has_the_bits_of_its_own_kernel(M, K):
    """A row's result is the same whether its norm is folded in (steps of up to 16 rows) or a kernel of its own (longer steps)."""
    gen = torch.Generator().manual_seed(K + M)
    x = (torch.randn(M, K, generator=gen) * torch.exp(2.0 * torch.randn(M, K, generator=gen))).to(DEV)
    norm, w = (1.0 + 0.3 * torch.randn(K, generator=gen)).to(DEV), torch.randn(24, K, generator=gen).to(DEV)
    normed, got, want = torch.empty_like(x), torch.empty(M, 24, device=DEV), torch.empty(M, 24, device=DEV)
    check(native.lib().celeg_rmsnorm(ptr(x), 0, None, 0, ptr(norm), ptr(normed), 0, None, M, K, ctypes.c_float(1e-5), 0, None))
    check(native.lib().celeg_gemm_f32(ptr(normed), K, ptr(w), K, None, ptr(want), 24, M, 24, K, None))
    check(call(x, w, got, 24, STORE, norm))
    assert torch.equal(got, want)
    # the other ends: the convolution of one tap of 1 multiplies the streams, SwiGLU is a row's own
    out, one = torch.empty(M, 8, device=DEV), torch.empty(1, 12, device=DEV)
    conv = (torch.ones(8, 1, device=DEV), None, torch.zeros(M, 1, 8, device=DEV), torch.arange(M, dtype=torch.int32, device=DEV))
    check(call(x, w, out, 8, CONV, norm, None, conv))
    streams = want.view(M, 3, 8)
    assert torch.equal(out, streams[:, 1] * (streams[:, 0] * streams[:, 2]))
    out = torch.empty(M, 12, device=DEV)
    check(call(x, w, out, 12, SWIGLU, norm))
    check(call(x[M - 1:], w, one, 12, SWIGLU, norm))
    assert torch.equal(one[0], out[M - 1])


def one_layer_of_each(folder, width, bias=False):
    """A model of a short convolution's and an attention's layer, float32."""
    from celeg_amd.weights import write_random_model
    config = {"architectures": ["Lfm2ForCausalLM"], "vocab_size": 256, "hidden_size": width, "num_hidden_layers": 2,
              "layer_types": ["conv", "full_attention"], "num_attention_heads": width // 32, "num_key_value_heads": width // 64,
              "head_dim": 32, "intermediate_size": 320, "block_auto_adjust_ff_dim": False, "rope_theta": 10000.0, "conv_L_cache": 3,
              "conv_bias": bias, "tie_word_embeddings": True, "norm_eps": 1e-5, "max_position_embeddings": 128, "eos_token_id": 7}
    return write_random_model(config, str(folder), seed=width, dtype=torch.float32, std=0.03)


@pytest.mark.parametrize("width,bias", [(256, True), (640, False), (1024, True)])
def test_logits_with_and_without(tmp_path, width, bias):
    """Steps of 7, 16, 9 and 1 rows with the folded products (their path counts them) and without (it does not): the same bits, near 64 bits."""
    from celeg_amd.engine import StepEntry, load_model
    folder = one_layer_of_each(tmp_path, width, bias)
    cfg, W = plain.load_model_folder(folder)
    tokens = random_tokens(cfg["vocab_size"], 40, seed=3)
    ref = plain.model_logits(cfg, W, tokens).double()
    got = {}
    for fused in (1, 0):
        lm = load_model(folder, dtype="float32", page_tokens=16, n_pages=16, max_requests=2, max_batched_tokens=64)
        lm.set_knob("use_fused", fused)
        slot, rows = lm.cache.open(), []
        for first, n in [(0, 7), (7, 16), (23, 9)] + [(i, 1) for i in range(32, 40)]:
            assert lm.cache.prepare(slot, first, n)
            rows.append(lm.runner.step([StepEntry(slot, first, tokens[first:first + n], [n - 1])])[0].double())
        assert (lm.paths()["linear_f32_fused"] > 0) == bool(fused)
        got[fused], want = torch.stack(rows), ref[[6, 22] + list(range(31, 40))]
        assert float((got[fused] - want).norm() / want.norm()) <= 2e-6
        lm.close()
    assert torch.equal(got[1], got[0])


@pytest.mark.parametrize("width,folded", [(192, False), (256, True), (1024, True), (1088, False), (2048, False)])
def test_which_streams_are_folded(tmp_path, width, folded):
    """Up to 16 rows of streams 256 to 1,024 wide: four products of each layer; other streams and more rows none.  A row's logits are the
    same beside 0, 15 and 16 other tokens."""
    from celeg_amd.engine import StepEntry, load_model
    folder = one_layer_of_each(tmp_path, width)
    cfg, W = plain.load_model_folder(folder)
    tokens = random_tokens(cfg["vocab_size"], 34, seed=4)
    ref = plain.model_logits(cfg, W, tokens).double()
    lm = load_model(folder, dtype="float32", page_tokens=16, n_pages=16, max_requests=2, max_batched_tokens=64)
    lm.set_knob("use_graphs", 0)
    slot, rows = lm.cache.open(), []
    for first, n in ((0, 16), (16, 17), (33, 1)):
        before = lm.paths()["linear_f32_fused"]
        assert lm.cache.prepare(slot, first, n)
        rows.append(lm.runner.step([StepEntry(slot, first, tokens[first:first + n], [n - 1])])[0].double())
        assert lm.paths()["linear_f32_fused"] - before == (8 if folded and n <= 16 else 0)
    got, want = torch.stack(rows), ref[[15, 32, 33]]
    assert float((got - want).norm() / want.norm()) <= 2e-6
    last = []
    for sizes in ((16, 17), (16, 16, 1), (17, 16), (1, 15, 17)):         # position 32 ends a portion of 17, 1, 16 and 17
        slot, at = lm.cache.open(), 0
        for n in sizes:
            assert lm.cache.prepare(slot, at, n)
            out = lm.runner.step([StepEntry(slot, at, tokens[at:at + n], [n - 1])])[0].clone()
            at += n
        last.append(out)
        lm.cache.close(slot)
    assert all(torch.equal(x, last[0]) for x in last)
    lm.close()
