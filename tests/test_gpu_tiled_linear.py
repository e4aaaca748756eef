"""The fused bfloat16 products for many rows (gemm_tiles.hip) alone, against torch: every
epilogue, every tile shape, at sizes that are no multiple of the tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16
N_SHAPES = 12


@pytest.fixture(scope="module")
def ops():
    from kernel_ops import HipOps
    ops = HipOps(DEV)
    yield ops
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(-1)


def randn(*shape, seed=0, scale=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def product(a, w, scale=None, bias=None):
    y = a.double() @ w.double().T
    if scale is not None:
        y = y * scale.double()[:, None]
    if bias is not None:
        y = y + bias.double()
    return y


def bf16_round(x):
    return x.to(torch.float32).to(BF).double()


# (the last: more blocks of k than any shape has stages, on sizes that are no whole number of tiles)
SIZES = [(300, 200, 128), (65, 36, 64), (512, 256, 192), (129, 1024, 1024), (520, 648, 192), (333, 396, 640)]


def test_every_shape_is_tested(ops):
    assert ops._lib("gemm_tiles").celeg_gemm_tiles_shapes() == N_SHAPES


@pytest.mark.parametrize("shape", list(range(N_SHAPES)) + [-1])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_store_with_row_scale_and_bias(ops, shape, M, N, K):
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(shape)
    a = randn(M, K, seed=1, dtype=BF)
    w = randn(N, K, seed=2, scale=0.05, dtype=BF)
    bias = randn(N, seed=3) if shape % 2 else None
    eps, blocks = 1e-5, 11                       # more partial sums than one round of loads
    g = torch.Generator().manual_seed(4)
    stats = (torch.rand(M, blocks + 2, generator=g) * K / blocks).to(DEV)
    scale = 1.0 / torch.sqrt(stats[:, :blocks].sum(1) / K + eps)
    out = torch.zeros(M + 1, N, dtype=BF, device=DEV)
    ops.tiled_linear(a, w, out[:M], bias=bias, stats=stats, stat_blocks=blocks, eps=eps)
    ref = product(a, w, scale, bias)
    assert float((out[:M].double() - ref).abs().max()) <= 2 ** -7 * float(ref.abs().max())
    assert float(out[M].abs().max()) == 0        # nothing behind the last row is written
    # without statistics the sums are stored as they are
    ops.tiled_linear(a, w, out[:M], bias=bias)
    ref = product(a, w, None, bias)
    assert float((out[:M].double() - ref).abs().max()) <= 2 ** -7 * float(ref.abs().max())


@pytest.mark.parametrize("shape", list(range(N_SHAPES)) + [-1])
@pytest.mark.parametrize("M,ff,K", SIZES)
def test_swiglu(ops, shape, M, ff, K):
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(shape)
    a = randn(M, K, seed=5, dtype=BF)
    w = randn(2 * ff, K, seed=6, scale=0.1, dtype=BF)
    bias = randn(2 * ff, seed=7, scale=0.1) if shape % 2 else None
    y = product(a, w, None, bias)
    gate, up = bf16_round(y[:, :ff]), bf16_round(y[:, ff:])
    ref = gate / (1 + torch.exp(-gate)) * up
    out = torch.zeros(M, ff, dtype=BF, device=DEV)
    ops.tiled_linear(a, w, out, epilogue="swiglu", bias=bias)
    # a flip of the rounding of gate or up moves the result by one bfloat16 step of it
    bound = 2 ** -6 * float(ref.abs().max()) + 2 ** -7 * float((up.abs() * (1 + gate.abs())).max())
    assert float((out.double() - ref).abs().max()) <= bound


def swiglu_of(ops, gates, ups):
    """What the SwiGLU epilogue makes of every pair of a gate and an up value: each is one product with 1."""
    M, N, K = len(gates), len(ups), 64
    a, w = torch.zeros(M, K, dtype=BF), torch.zeros(2 * N, K, dtype=BF)
    a[:, 0], a[:, 1], w[:N, 0], w[N:, 1] = gates, 1.0, 1.0, ups
    out = torch.empty(M, N, dtype=BF, device=DEV)
    ops.tiled_linear(a.to(DEV), w.to(DEV), out, epilogue="swiglu")
    return out.cpu()


@pytest.mark.parametrize("shape", [0, 9, 10, 11])
def test_swiglu_of_every_gate(ops, shape):
    """Every normal gate, those whose 1 + e^-g has a reciprocal below the normal numbers among them."""
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(shape)
    gates = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(BF)
    gates = gates[torch.isfinite(gates) & ((gates.abs() >= 2.0 ** -126) | (gates == 0))]
    ups = torch.tensor([1.0, -1.4453125, 0.75, 1.9921875] + [2.0 ** k for k in range(-10, 10)], dtype=BF)
    got, g = swiglu_of(ops, gates, ups).double(), gates.double()
    want = torch.where(g < -700, torch.zeros_like(g), g / (1 + torch.exp(-g.clamp(min=-700))))[:, None] * ups.double()
    # the rounding to bfloat16, the exponential's error (|g| 2^-24 from its argument, an ulp of its own) and three roundings; where
    # e^-g is beyond 32-bit (below -88.7) the result is 0, what it should be then is below 2^-110 with these ups
    bound = want.abs() * (2.0 ** -8 + (g.abs().clamp(max=100.0)[:, None] + 8) * 2.0 ** -23) + 2.0 ** -126
    holds = ((got - want).abs() <= bound) | (want.abs() >= 2.0 ** 127)           # (there the product overflows)
    assert bool(holds[g >= -88.5].all())
    assert float(got[g < -88.75].abs().max()) == 0


@pytest.mark.parametrize("shape", [0, 9, 10, 11])
def test_swiglu_divides_as_32_bit_division_does(ops, shape):
    """The quotient is rounded correctly: where no error of the exponential within its bound can change 1 + e^-g, the result's
    bits follow from it (among them 5.9375, whose quotient lies beside the middle of two bfloat16 numbers)."""
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(shape)
    gates = torch.arange(0x3E00, 0x4190, dtype=torch.int32).to(torch.int16).view(BF)       # 0.125 .. 17.9
    ups = torch.arange(0x3F80, 0x4000, dtype=torch.int32).to(torch.int16).view(BF)         # every mantissa
    e = torch.exp(-gates.double())
    error = e * (gates.double() + 4) * 2.0 ** -23
    x = (1 + e).float()
    sure = ((1 + e - error).float() == x) & ((1 + e + error).float() == x)
    assert int(sure.sum()) > 200 and bool(sure[gates == 5.9375].all())
    want = ((gates.float() * (torch.ones_like(x) / x))[:, None] * ups.float()).to(BF)
    assert torch.equal(swiglu_of(ops, gates, ups)[sure], want[sure])


@pytest.mark.parametrize("shape", list(range(N_SHAPES)) + [-1])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_residual_adds_in_place_refreshes_the_copy_and_leaves_partial_sums(ops, shape, M, N, K):
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(shape)
    a = randn(M, K, seed=8, dtype=BF)
    w = randn(N, K, seed=9, scale=0.05, dtype=BF)
    bias = randn(N, seed=10) if shape % 2 else None
    h0 = randn(M + 1, N, seed=11)
    h = h0.clone()
    blocks = ops.tiled_stat_blocks(M, N, K)
    copy = torch.zeros(M, N, dtype=BF, device=DEV)
    sums = torch.zeros(M, blocks + 1, device=DEV)
    ops.tiled_linear(a, w, h[:M], epilogue="residual", bias=bias, out_bf16=copy, stats_out=sums)
    assert ops.last_stat_blocks == blocks
    y = product(a, w, None, bias)
    ref = h0[:M].double() + bf16_round(y)
    # the product enters the sum rounded to bfloat16: a flip of that rounding is one step of it
    assert float((h[:M].double() - ref).abs().max()) <= 2 ** -7 * float(y.abs().max())
    assert torch.equal(h[M], h0[M])
    assert torch.equal(copy, h[:M].to(BF))
    squares = (h[:M].double() ** 2).sum(1)
    assert float(((sums[:, :blocks].double().sum(1) - squares).abs() / squares).max()) < 1e-5
    assert float(sums[:, blocks].abs().max()) == 0


@pytest.mark.parametrize("M,N,K,blocks", [(2000, 1024, 2304, 16), (2000, 1024, 1024, 8), (2048, 2048, 1024, 16),
                                          (2048, 3072, 1024, 16), (1024, 3072, 1024, 16)])
def test_the_shapes_chosen_for_a_prefill(ops, M, N, K, blocks):
    """What the choice of shape gives at the sizes of a prefill of some 2,000 rows (few weight
    rows with a long and a short K, q/k/v, in_proj), against torch, with the residual epilogue;
    the number of tile columns says which shape it was."""
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(-1)
    assert ops.tiled_stat_blocks(M, N, K) == blocks
    a = randn(M, K, seed=20, dtype=BF)
    w = randn(N, K, seed=21, scale=0.03, dtype=BF)
    h0 = randn(M, N, seed=22)
    h = h0.clone()
    copy = torch.zeros(M, N, dtype=BF, device=DEV)
    sums = torch.zeros(M, blocks, device=DEV)
    ops.tiled_linear(a, w, h, epilogue="residual", out_bf16=copy, stats_out=sums)
    y = product(a, w)
    ref = h0.double() + bf16_round(y)
    assert float((h.double() - ref).abs().max()) <= 2 ** -7 * float(y.abs().max())
    assert torch.equal(copy, h.to(BF))
    squares = (h.double() ** 2).sum(1)
    assert float(((sums.double().sum(1) - squares).abs() / squares).max()) < 1e-5


@pytest.mark.parametrize("shape", range(N_SHAPES))
def test_a_row_does_not_depend_on_the_other_rows(ops, shape):
    """The same row in a step of 70 rows and in one of 700 gives the same bits where the tile
    shape is the same (the sums of a row are formed in an order that K alone fixes)."""
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(shape)
    K, N = 192, 128
    a = randn(700, K, seed=12, dtype=BF)
    w = randn(N, K, seed=13, scale=0.05, dtype=BF)
    big = torch.empty(700, N, dtype=BF, device=DEV)
    small = torch.empty(70, N, dtype=BF, device=DEV)
    ops.tiled_linear(a, w, big)
    ops.tiled_linear(a[330:400], w, small)
    assert torch.equal(big[330:400], small)


def test_unsupported_sizes_are_refused(ops):
    from kernel_ops import KernelError
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(-1)
    a = randn(80, 96, dtype=BF)
    with pytest.raises(KernelError):             # inner size no multiple of 64
        ops.tiled_linear(a, randn(64, 96, dtype=BF), torch.empty(80, 64, dtype=BF, device=DEV))
    a = randn(80, 128, dtype=BF)
    with pytest.raises(KernelError):             # columns no multiple of 4
        ops.tiled_linear(a, randn(66, 128, dtype=BF), torch.empty(80, 66, dtype=BF, device=DEV))
    with pytest.raises(KernelError):             # a 32-bit output goes with the residual epilogue only
        ops.tiled_linear(a, randn(64, 128, dtype=BF), torch.empty(80, 64, device=DEV))
    with pytest.raises(KernelError):
        ops.tiled_linear(a, randn(64, 128, dtype=BF), torch.empty(80, 64, dtype=BF, device=DEV),
                         stats_out=torch.empty(80, 4, device=DEV))
    assert not ops.tiled_linear_ok(80, 64, 96)
    assert ops.tiled_linear_ok(80, 64, 128, 4608)


@pytest.mark.parametrize("M", [65, 256, 257, 513, 700, 1000, 1300, 2048, 2049])
@pytest.mark.parametrize("N,K", [(1024, 4608), (1024, 1024), (3072, 64), (264, 128)])
def test_a_row_is_the_same_in_every_chosen_tile(ops, M, N, K):
    """Every tile that the rule picks over these rows sums a row's products in one order: the bits of a step's
    last 65 rows are those of a step of these rows alone, for a plain product and behind the SwiGLU."""
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(-1)
    a = randn(M, K, seed=12, dtype=BF)
    w = randn(N, K, seed=13, scale=0.05, dtype=BF)
    for epilogue, columns in (("store", N), ("swiglu", N // 2)):
        big = torch.zeros(M + 1, columns, dtype=BF, device=DEV)
        small = torch.empty(65, columns, dtype=BF, device=DEV)
        ops.tiled_linear(a, w, big[:M], epilogue=epilogue)
        ops.tiled_linear(a[M - 65:], w, small, epilogue=epilogue)
        assert torch.equal(big[M - 65:M], small) and float(big[M].abs().max()) == 0
    ref = product(a, w)
    out = torch.empty(M, N, dtype=BF, device=DEV)
    ops.tiled_linear(a, w, out)
    assert float((out.double() - ref).abs().max()) <= 2 ** -7 * float(ref.abs().max())


@pytest.mark.parametrize("M,N,K,blocks", [
    (1500, 1024, 1984, 8), (1500, 1024, 2048, 16),             # 64x128; 128x64 from 2,048 values of k on
    (1024, 3072, 128, 16), (1089, 3072, 128, 24),              # 64x192 while it fits, then 128 columns
    (3000, 1024, 64, 8)])
def test_where_the_choice_of_shape_changes(ops, M, N, K, blocks):
    ops._lib("gemm_tiles").celeg_gemm_tiles_force(-1)
    assert ops.tiled_stat_blocks(M, N, K) == blocks
    a, w = randn(M, K, seed=24, dtype=BF), randn(N, K, seed=25, scale=0.03, dtype=BF)
    out, ref = torch.empty(M, N, dtype=BF, device=DEV), product(a, w)
    ops.tiled_linear(a, w, out)
    assert float((out.double() - ref).abs().max()) <= 2 ** -7 * float(ref.abs().max())


# ---------------------------------------------------------------- the q/k/v product with its tail
@pytest.mark.parametrize("K", [128, 1024])
@pytest.mark.parametrize("lengths", [[333, 131, 1, 97], [803, 131, 1, 166], [1990, 131, 1, 166]])
def test_qkv_product_on_larger_tiles(ops, lengths, K):
    """As below, on steps of as many rows as take the tiles of 64x128 and of 128x128 (one and two a compute unit),
    with fewer blocks of k than stages and with more."""
    check_qkv_product(ops, 16, 8, K, True, True, [0, 5, 130, 77], lengths)


@pytest.mark.parametrize("heads,kv_heads,K,rotate,normed", [(16, 8, 1024, True, True), (6, 2, 192, True, False),
                                                            (4, 4, 128, False, True), (3, 1, 64, True, True)])
def test_qkv_product_with_norm_rotation_and_cache_write(ops, heads, kv_heads, K, rotate, normed):
    check_qkv_product(ops, heads, kv_heads, K, rotate, normed, [0, 5, 130, 77], [203, 131, 1, 66])


def check_qkv_product(ops, heads, kv_heads, K, rotate, normed, starts, lengths):
    """The product of the q, k and v projections that normalises and turns the query and key
    heads and writes keys and values into the pages inside its own kernel, against the product
    followed by qk_norm_rope_store: a step of three requests (portions that start at positions
    0, 5 and 130, so that groups of four rows start on a multiple of four, in the middle of one,
    and straddle the border between two requests; one request brings a single row).  Values must
    come out bit for bit; queries and keys may differ by a rounding (the sums of squares are
    added in another order)."""
    import plain_lfm2 as plain
    from celeg_amd.engine import StepEntry
    from kernel_harness import build_batch, make_cache
    hd, n_layers, layer, page_tokens = 64, 2, 1, 16
    total = sum(lengths)
    N = (heads + 2 * kv_heads) * hd
    a = randn(total, K, seed=30, dtype=BF)
    w = randn(N, K, seed=31, scale=0.05, dtype=BF)
    bias = randn(N, seed=32) if not normed else None
    qw = (1 + randn(hd, seed=33, scale=0.2)) if normed else None
    kw = (1 + randn(hd, seed=34, scale=0.2)) if normed else None
    inv_freq = torch.tensor(plain.rope_inverse_frequencies(10000.0, hd), dtype=torch.float64).float().to(DEV) if rotate else None
    eps, blocks = 1e-5, 5
    g = torch.Generator().manual_seed(35)
    stats = (torch.rand(total, blocks, generator=g) * K / blocks).to(DEV)
    results = []
    for fused in (False, True):
        cache = make_cache(kv_heads, hd, n_layers, BF, page_tokens=page_tokens, n_pages=64 + sum(lengths) // page_tokens, max_context=2048, slots=4)
        kv = cache.layer_cache(layer).kv
        slots = [cache.open() for _ in lengths]
        entries = []
        for slot, start, n in zip(slots, starts, lengths):
            assert cache.prepare(slot, 0, start + n)
            entries.append(StepEntry(slot, start, [0] * n))
        batch, keep = build_batch(ops, cache, entries)
        qkv = torch.zeros(total + 1, N, dtype=BF, device=DEV)
        if fused:
            ops.tiled_linear(a, w, qkv[:total], stats=stats, stat_blocks=blocks, eps=eps, bias=bias,
                             qkv=dict(heads=heads, kv_heads=kv_heads, q_weight=qw, k_weight=kw, eps=1e-6, inv_freq=inv_freq,
                                      batch=batch, kv=kv))
        else:
            ops.tiled_linear(a, w, qkv[:total], stats=stats, stat_blocks=blocks, eps=eps, bias=bias)
            q, k, v = qkv[:total, :heads * hd], qkv[:total, heads * hd:(heads + kv_heads) * hd], qkv[:total, (heads + kv_heads) * hd:]
            ops.qk_norm_rope_store(q, k, v, qw, kw, 1e-6, inv_freq, hd, heads, kv_heads, hd, batch, kv)
        torch.cuda.synchronize()
        assert float(qkv[total].abs().max()) == 0
        table = kv.table.cpu()
        pages = [int(table[slot, p]) for slot, start, n in zip(slots, starts, lengths)
                 for p in range((start + n + page_tokens - 1) // page_tokens)]
        others = sorted(set(range(kv.k.shape[0])) - set(pages))
        assert float(kv.k[others].float().abs().max()) == 0 and float(kv.v[others].float().abs().max()) == 0
        assert float(kv.k[:, 0].float().abs().max()) == 0          # the other layer's pages
        results.append((qkv[:total, :heads * hd].float().clone(), kv.k[pages].float().clone(), kv.v[pages].clone()))
    (qa, ka, va), (qb, kb, vb) = results
    assert torch.equal(va, vb) and float(va.float().abs().max()) > 0
    for x, y in ((qa, qb), (ka, kb)):
        assert float(x.abs().max()) > 0
        # a rounding of bfloat16 where the two differ at all
        assert float(((x - y).abs() / (x.abs() + y.abs() + 1e-3)).max()) <= 2 ** -7
        assert float((x != y).float().mean()) < 0.02
