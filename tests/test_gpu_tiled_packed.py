"""The tiled products into the residual stream from packed weights ([K/32, rows, 32]), and with K cut over workgroups."""
import pytest
import torch

from kernel_ops import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    return HipOps()


def randn(*shape, seed, scale=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(dtype).to(DEV)


def packed_weight(ops, w):
    return ops.fold_weight(w, None, packed=True)


@pytest.mark.parametrize("shape", [0, 1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("M,N,K", [(1, 4, 64), (33, 68, 192), (130, 200, 320), (257, 132, 1088)])
def test_packed_weights_give_the_bits_of_weights_as_they_are(ops, shape, M, N, K):
    """Every tile that takes packed weights, K a whole number of blocks but not of stages, rows and columns that end inside tiles."""
    a, w, h0 = randn(M, K, seed=41, dtype=BF), randn(N, K, seed=42, scale=0.05, dtype=BF), randn(M + 1, N, seed=43)
    results = []
    for weight in (w, packed_weight(ops, w)):
        ops._lib("gemm_tiles").celeg_gemm_tiles_force(shape)
        h, copy, sums = h0.clone(), torch.zeros(M, N, dtype=BF, device=DEV), torch.zeros(M, (N + 31) // 32 + 1, device=DEV)
        ops.tiled_linear(a, weight, h[:M], epilogue="residual", out_bf16=copy, stats_out=sums)
        ops._lib("gemm_tiles").celeg_gemm_tiles_force(-1)
        results.append((h, copy, sums))
    for x, y in zip(*results):
        assert torch.equal(x, y)
    assert torch.equal(results[1][0][M], h0[M])


@pytest.mark.parametrize("shape,slices", [(0, 2), (0, 4), (0, 5), (1, 2), (1, 4), (3, 3), (-1, 0)])
@pytest.mark.parametrize("M,N,K", [(1, 4, 320), (70, 1024, 4608), (130, 200, 4160), (300, 260, 4096)])
def test_k_over_several_workgroups(ops, shape, slices, M, N, K):
    """Tiles whose K is cut (slices of unlike lengths among them), by force and by the rule: the 64-bit product, the same bits
    in every launch (the counts are zeros again behind each), the stream's copy and its rows' squares."""
    lib = ops._lib("gemm_tiles")
    a, w, h0 = randn(M, K, seed=44, dtype=BF), randn(N, K, seed=45, scale=0.05, dtype=BF), randn(M + 1, N, seed=46)
    weight, bias = packed_weight(ops, w), randn(N, seed=47)
    y = a.double() @ w.double().t() + bias.double()
    lib.celeg_gemm_tiles_force(shape)
    lib.celeg_gemm_tiles_force_slices(slices)
    results = []
    try:
        for _ in range(3):
            h, copy, sums = h0.clone(), torch.zeros(M, N, dtype=BF, device=DEV), torch.zeros(M, (N + 31) // 32 + 1, device=DEV)
            ops.tiled_linear(a, weight, h[:M], epilogue="residual", bias=bias, out_bf16=copy, stats_out=sums)
            results.append((h, copy, sums))
    finally:
        lib.celeg_gemm_tiles_force(-1)
        lib.celeg_gemm_tiles_force_slices(0)
    h, copy, sums = results[0]
    # the product is rounded to bfloat16 ahead of the sum: half a step of it, and K 32-bit additions of terms as large as |a||w|
    bound = y.abs() * 2.0 ** -8 + (a.abs().double() @ w.abs().double().t()) * K * 2.0 ** -24 + 1e-5
    assert bool(((h[:M].double() - h0[:M].double() - y).abs() <= bound + h[:M].abs().double() * 2.0 ** -23).all())
    assert torch.equal(copy, h[:M].to(BF)) and torch.equal(h[M], h0[M])
    ssq = (h[:M].double() ** 2).sum(1)
    assert bool(((sums.double().sum(1) - ssq).abs() <= ssq * 1e-5).all())
    for other in results[1:]:
        for x, z in zip(results[0], other):
            assert torch.equal(x, z)


def test_where_packed_weights_are_taken(ops):
    lib = ops._lib("gemm_tiles")
    taken = lambda M, N, K: bool(lib.celeg_gemm_tiles_packed(M, N, K))
    assert taken(65, 1024, 4608) and taken(640, 1024, 4608) and taken(2048, 1024, 4608)
    assert not taken(1300, 1024, 4608) and not taken(1000, 2048, 8192)
