"""Tiled products beyond one round of workgroups (the tile of 256x256 among those chosen)."""
import pytest
import torch

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
