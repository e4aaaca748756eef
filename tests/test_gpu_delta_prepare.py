"""What the delta rule reads (convolution, silu, unit norms, beta and decay) by the kernel with four channels a lane, against the one
with a wavefront a row and head (which rows at any distance take)."""
import ctypes

import pytest
import torch

from kernel_ops import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("G,H,D,V,taps,decay", [(8, 16, 64, 64, 4, True), (1, 1, 16, 4, 1, True), (2, 6, 32, 20, 2, False), (3, 3, 128, 128, 3, True),
                                                (1, 2, 256, 12, 4, True)])
@pytest.mark.parametrize("lengths", [(256,), (1, 2, 3, 1, 270, 2), (229, 66)])
def test_quads(dtype, G, H, D, V, taps, decay, lengths):
    lib = HipOps()._lib("delta_rule")
    T, C = sum(lengths), 2 * G * D + H * V
    gen = torch.Generator().manual_seed(T + C)

    def randn(*shape):
        return torch.randn(*shape, generator=gen).to(DEV)
    width = C + 8 + 2 * ((H + 3) // 4 * 4)
    data = randn(T, width).to(dtype)
    conv_w, saved = randn(C, taps), randn(len(lengths) + 1, max(taps - 1, 1), C)
    a_log, dt_bias = randn(H), randn(H)
    starts = [7 * (i % 2) for i in range(len(lengths))]
    ints = {"positions": [s + i for s, n in zip(starts, lengths) for i in range(n)], "token_seq": [j for j, n in enumerate(lengths) for _ in range(n)],
            "seq_start": starts, "token_slot": [len(lengths) - j for j, n in enumerate(lengths) for _ in range(n)]}
    ints = {k: torch.tensor(v, dtype=torch.int32, device=DEV) for k, v in ints.items()}
    p = ctypes.c_void_p
    results = []
    for odd in (1, 0):
        proj = torch.zeros(T, width + odd, dtype=dtype, device=DEV)
        proj[:, :width] = data
        qk, v, bd = torch.full((T + 1, 2 * G * D), 7.0, device=DEV), torch.full((T + 1, H * V), 7.0, device=DEV), torch.full((T + 1, 2 * H), 7.0, device=DEV)
        rc = lib.celeg_delta_prepare(p(proj.data_ptr()), width + odd, 0 if dtype == torch.float32 else 1, C + 8, C + 8 + (H + 3) // 4 * 4, p(conv_w.data_ptr()),
                                     p(a_log.data_ptr() if decay else None), p(dt_bias.data_ptr() if decay else None), p(saved.data_ptr()),
                                     ctypes.c_size_t(saved.stride(0)), *(p(ints[k].data_ptr()) for k in ("positions", "token_seq", "seq_start", "token_slot")),
                                     p(qk.data_ptr()), p(v.data_ptr()), p(bd.data_ptr()), T, G, H, D, V, taps, p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        torch.cuda.synchronize()
        assert all(bool((x[T] == 7).all()) for x in (qk, v, bd))
        results.append((qk, v, bd))
    (qa, va, ba), (qb, vb, bb) = results
    assert torch.equal(va, vb) and torch.equal(ba, bb)
    # (a head of more than 64 values adds its squares in another order: some 2^-22 of up to 256 positive numbers)
    assert D > 64 or torch.equal(qa, qb)
    assert float((qa - qb).abs().max()) <= 4e-7 * float(qa.abs().max())
