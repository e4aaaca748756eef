"""Attention over compressed rows on the matrix cores, called as the host code calls it: sizes of a row at the edges of the three
that the kernel is built for, portions and single tokens, contexts at the edges of a block of keys, against 64 bits."""
import ctypes
import math

import pytest
import torch

from celeg_amd import native
from test_gpu_single_tokens import check, ints, ptr

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


# (rank, rotated): the largest of each size and the smallest of the next, ranks that fill no pair of tiles, rows shorter than a step
SIZES = [(16, 0), (16, 8), (128, 32), (128, 40), (144, 16), (112, 0), (256, 32), (256, 40), (272, 16), (512, 64)]


@pytest.mark.parametrize("exact", [0, 1])
@pytest.mark.parametrize("window", [0, 1, 65, 200])
@pytest.mark.parametrize("rank,rot", SIZES)
def test_rows_and_single_tokens_against_64_bits(rank, rot, window, exact):
    D, H, page, layers, layer = rank + rot, 3 if rank > 128 else 17, 16, 2, 1
    seqs = [(1, 0), (1, 63), (1, 64), (1, 400), (2, 62), (64, 0), (65, 127), (130, 3)]        # (rows, tokens before them)
    gen = torch.Generator().manual_seed(rank + rot + window)
    T, n, singles = sum(k for k, _ in seqs), len(seqs), 4
    per = (max(k + s for k, s in seqs) + page - 1) // page
    pages = torch.randperm(n * per, generator=gen).int().view(n, per)
    pool = torch.randn(n * per, layers, page, D, generator=gen).to(BF)
    for i, (k, s) in enumerate(seqs):             # what lies behind a request's last key may be anything
        if (k + s) % page:
            pool[int(pages[i, (k + s) // page]), :, (k + s) % page:] = float("nan")
    pool, q = pool.to(DEV), torch.randn(T, H * D, generator=gen).to(BF).to(DEV)
    sink = torch.randn(H, generator=gen).to(DEV)
    cu = [0]
    for k, _ in seqs:
        cu.append(cu[-1] + k)
    tokens = [(i, s + j) for i, (k, s) in enumerate(seqs) for j in range(k)]
    out = torch.full((T, H * rank), 7.0, dtype=BF, device=DEV)
    splits, per_split, scale = 4, 2, 1.5 / math.sqrt(D)
    parts_o = torch.empty(singles * H * splits * rank, device=DEV)
    parts_ml = torch.empty(singles * H * splits * 2, device=DEV)
    table, d_cu, d_slot, d_start = pages.to(DEV), ints(cu), ints(list(range(n))), ints([s for _, s in seqs])
    d_token_slot, d_pos = ints([i for i, _ in tokens]), ints([p for _, p in tokens])
    for form, count, tiles in ((1, singles, 0), (0, 0, (T - singles) // 64 + n - singles)):
        check(native.lib().celeg_latent_attention_fast(
            form, ptr(q), H * D, ptr(pool), ptr(table), per, ptr(d_cu), ptr(d_slot), ptr(d_start), n, tiles, ptr(d_token_slot),
            ptr(d_pos), count, ptr(sink), ptr(out), H * rank, ptr(parts_o), ptr(parts_ml), splits, per_split, H, rank, rot, page, layers,
            layer, ctypes.c_float(scale), window, exact, None))
    torch.cuda.synchronize()
    got = out.double().cpu().view(T, H, rank)
    for i, (k, s) in enumerate(seqs):
        rows = pool[pages[i].long().to(DEV), layer].reshape(-1, D)[:k + s].double().cpu()
        at, keys = torch.arange(s, s + k)[:, None], torch.arange(k + s)[None]
        seen = (keys <= at) & ((at - keys < window) if window else True)
        scores = (q[cu[i]:cu[i + 1]].double().cpu().view(k, H, D).transpose(0, 1) @ rows.T) * scale
        scores = scores.masked_fill(~seen, -math.inf)
        weights = torch.softmax(torch.cat([scores, sink.double().cpu()[:, None, None].expand(-1, k, 1)], -1), -1)[..., :-1]
        want = (weights @ rows[:, :rank]).transpose(0, 1)
        # the result is rounded to bfloat16 (8 significant bits: half a unit of the last is 2^-8 of the value at most), each weight
        # too unless it enters as two numbers (so 2^-8 of the largest value at most); scores are 32-bit sums of up to 576 products
        bound = 2.0 ** -8 * want.abs() + (2.0 ** -8 if not exact else 0.0) * rows.abs().max() + 1e-4
        error = (got[cu[i]:cu[i + 1]] - want).abs()
        assert (error <= 1.05 * bound).all(), (i, (error / bound).max())



@pytest.mark.parametrize("single", [True, False])
def test_pages_of_more_values_than_32_bits_count(single):
    """A page of 4,096 tokens and 1,822 layers of 576 values is 4.3 G values (8.6 GB): the rows of the last of three pages and the
    last layer are read where they lie.  The same bits as from a pool of small pages."""
    rank, rot, H, page, layers = 512, 64, 3, 4096, 1822
    D = rank + rot
    if torch.cuda.mem_get_info()[0] < (40 << 30):
        pytest.skip("no room for three pages of 8.6 GB")
    context, rows_new = page + 64, 1 if single else 70
    big = torch.empty(3 * layers * page * D, dtype=BF, device=DEV)
    gen = torch.Generator().manual_seed(5)
    rows = torch.randn(context, D, generator=gen).to(BF).to(DEV)
    table_big = ints([2, 1])
    for i, p in enumerate((2, 1)):
        part = rows[i * page:(i + 1) * page]
        start = (p * layers + layers - 1) * page * D
        big[start:start + part.numel()] = part.reshape(-1)
    small_page = 16
    per = (context + small_page - 1) // small_page
    small = torch.zeros(per, small_page, D, dtype=BF, device=DEV)
    small.view(-1, D)[:context] = rows
    table_small = ints(list(range(per)))
    q = torch.randn(rows_new, H * D, generator=gen).to(BF).to(DEV)
    cu, slot, start, token_slot = ints([0, rows_new]), ints([0]), ints([context - rows_new]), ints([0] * rows_new)
    positions = ints(list(range(context - rows_new, context)))
    splits, per_split, scale = 4, 17, 1.5 / math.sqrt(D)
    parts_o, parts_ml = torch.empty(H * splits * rank, device=DEV), torch.empty(H * splits * 2, device=DEV)

    def run(pool, table, table_stride, page_tokens, n_layers):
        out = torch.full((rows_new, H * rank), 7.0, dtype=BF, device=DEV)
        check(native.lib().celeg_latent_attention_fast(
            1 if single else 0, ptr(q), H * D, ptr(pool), ptr(table), table_stride, ptr(cu), ptr(slot), ptr(start), 1, 0 if single else 2,
            ptr(token_slot), ptr(positions), 1 if single else 0, None, ptr(out), H * rank, ptr(parts_o), ptr(parts_ml), splits, per_split, H,
            rank, rot, page_tokens, n_layers, n_layers - 1, ctypes.c_float(scale), 0, 1, None))
        torch.cuda.synchronize()
        return out

    assert torch.equal(run(big, table_big, 2, page, layers), run(small, table_small, per, small_page, 1))
    assert native.lib().celeg_latent_attention_fast_ok(rank, rot, layers, page) == 1
    assert native.lib().celeg_latent_attention_fast_ok(rank, rot, layers * 8, page) == 0        # what the kernel's 32 bits do not hold
