"""Rotation of a part of a head by the kernel with four values a lane, against the kernel with a wavefront a head (which takes keys
whose rows lie at any distance) and against 64 bits."""
import pytest
import torch

import plain_lfm2 as plain
from kernel_harness import build_batch, make_cache
from kernel_ops import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,kv_heads,head_dim,rotary", [(16, 8, 64, 32), (2, 1, 64, 8), (6, 3, 64, 24), (5, 5, 64, 56), (4, 2, 64, 64),
                                                            (4, 2, 32, 8), (4, 2, 32, 24), (10, 5, 128, 64), (2, 1, 128, 120), (4, 2, 64, 12)])
@pytest.mark.parametrize("lengths", [(1, 1, 1), (3, 1, 66), (2050, 700)])
def test_part_of_a_head(dtype, heads, kv_heads, head_dim, rotary, lengths):
    from celeg_amd.engine import StepEntry
    ops, n, kvw = HipOps(), sum(lengths), kv_heads * head_dim
    gen = torch.Generator().manual_seed(rotary + n)

    def randn(*shape):
        return torch.randn(*shape, generator=gen)
    qw, kw = (1 + 0.1 * randn(head_dim)).to(DEV), (1 + 0.1 * randn(head_dim)).to(DEV)
    inv_freq = torch.tensor(plain.rope_inverse_frequencies(500000.0, rotary), dtype=torch.float64).float().to(DEV)
    q0, k0, v0 = randn(n, heads * head_dim).to(dtype).to(DEV), randn(n, kvw).to(dtype).to(DEV), randn(n, kvw).to(dtype).to(DEV)
    results = []
    for apart in (False, True):
        cache = make_cache(kv_heads, head_dim, 2, dtype, page_tokens=16, n_pages=n // 16 + 8, max_context=2080, slots=8)
        kv = cache.layer_cache(1).kv
        entries = []
        for length in lengths:
            slot = cache.open()
            assert cache.prepare(slot, 0, 5) and cache.prepare(slot, 5, length)
            entries.append(StepEntry(slot, 5, [0] * length))
        batch, keep = build_batch(ops, cache, entries)
        k = torch.zeros(n, kvw + 2, dtype=dtype, device=DEV)[:, :kvw] if apart else torch.zeros(n, kvw, dtype=dtype, device=DEV)
        k.copy_(k0)
        q = q0.clone()
        ops.qk_norm_rope_store(q, k, v0, qw, kw, 1e-5, inv_freq, rotary, heads, kv_heads, head_dim, batch, kv)
        torch.cuda.synchronize()
        order = batch.entry_order
        if not apart:
            positions = [5 + i for j in order for i in range(lengths[j])]
            cos, sin = plain.rope_cos_sin(positions, 500000.0, rotary)
            ref = plain.rope_apply(plain.head_rmsnorm(q0.double().cpu().reshape(n, heads, head_dim), qw.cpu(), 1e-5), cos, sin)
            # (angles are 32-bit products: 2^-24 of up to 2,055 radians)
            bound = 4e-3 if dtype == torch.bfloat16 else 3e-4
            assert float((q.double().cpu().reshape(ref.shape) - ref).abs().max()) < bound * float(ref.abs().max())
        # what the pages hold of the rows: keys [token, head, value], values likewise
        table, held = kv.table.cpu(), []
        for e in entries:
            pages = table[e.slot, :(5 + len(e.tokens) + 15) // 16].long().to(DEV)
            keys = kv.k[pages, 1].permute(0, 2, 1, 3).reshape(-1, kv_heads, head_dim)
            values = kv.v[pages, 1].permute(0, 3, 1, 2).reshape(-1, kv_heads, head_dim)
            held.append(torch.cat([keys[5:5 + len(e.tokens)], values[5:5 + len(e.tokens)]], 1).float())
        results.append((q.float(), torch.cat(held)))
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2e-6
    for a, b in zip(*results):
        assert float(b.abs().max()) > 0
        assert float((a - b).abs().max()) <= ulp * float(b.abs().max())
