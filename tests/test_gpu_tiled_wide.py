"""The tile of 256x256, and tiled products beyond one round of workgroups by the tile that the rule chooses for them."""
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


@pytest.mark.gpu
@pytest.mark.parametrize("shape,M,N,K", [(11, 1, 4, 64), (11, 257, 132, 192), (11, 255, 256, 320), (11, 300, 516, 1088)])
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


# (7: 128x192, 8: 128x128 with two workgroups a compute unit, 9: 256x192, 10: 256x288, 11: 256x256; both sides of SwiGLU's N)
@pytest.mark.gpu
@pytest.mark.parametrize("epilogue,M,N,K,chosen", [
    ("swiglu", 440, 4608, 512, 7), ("swiglu", 440, 4608, 64, 8), ("swiglu", 928, 4608, 128, 9), ("swiglu", 1843, 4608, 128, 10),
    ("swiglu", 1294, 4608, 512, 11), ("swiglu", 2047, 8192, 2048, 11), ("swiglu", 1200, 8192, 2048, 9),
    ("store", 1294, 3072, 512, 7), ("store", 1294, 3072, 64, 8), ("store", 2575, 3072, 128, 9), ("store", 3612, 4608, 128, 10),
    ("store", 4100, 3072, 512, 11), ("residual", 1294, 3072, 512, 7), ("residual", 1294, 3072, 64, 8), ("residual", 2575, 3072, 128, 9),
    ("residual", 3612, 4608, 128, 10), ("residual", 5137, 2052, 512, 11)])
def test_the_tile_that_the_rule_chooses(ops, epilogue, M, N, K, chosen):
    """The bits of the smallest tile, with a bias, and the partial sums of squares of what goes into the stream."""
    lib = ops._lib("gemm_tiles")
    lib.celeg_gemm_tiles_force(-1)
    assert lib.celeg_gemm_tiles_chosen(M, N, K, {"store": 0, "residual": 2, "swiglu": 3}[epilogue]) == chosen
    streams = 2 if epilogue == "swiglu" else 1
    a, w, bias = randn(M, K, seed=61, dtype=BF), randn(N * streams, K, seed=62, scale=0.1, dtype=BF), randn(N * streams, seed=63)
    results = []
    for force in (0, -1):
        lib.celeg_gemm_tiles_force(force)
        if epilogue == "residual":
            out, copy = torch.ones(M + 1, N, device=DEV), torch.zeros(M, N, dtype=BF, device=DEV)
            sums = torch.zeros(M, (N + 63) // 64 + 1, device=DEV)
            ops.tiled_linear(a, w, out[:M], epilogue=epilogue, bias=bias, out_bf16=copy, stats_out=sums)
            squares = (out[:M].double() ** 2).sum(1)
            assert float(((sums.double().sum(1) - squares).abs() / squares).max()) < 1e-5
            assert torch.equal(copy, out[:M].to(BF))
        else:
            out = torch.ones(M + 1, N, dtype=BF, device=DEV)
            ops.tiled_linear(a, w, out[:M], epilogue=epilogue, bias=bias, stats=randn(M, 4, seed=64).abs() + 0.1, stat_blocks=4, eps=1e-5)
        results.append(out)
    lib.celeg_gemm_tiles_force(-1)
    assert torch.equal(results[0], results[1]) and bool((results[1][M] == 1).all())
