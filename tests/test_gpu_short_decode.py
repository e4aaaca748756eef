"""Single tokens' attention on both sides of the number of keys up to which one workgroup takes a request and
key/value head whole: few requests (10 rounds of 64 keys) and 64 pairs of request and head (16 rounds)."""
from types import SimpleNamespace

import pytest
import torch

from kernel_harness import build_batch, make_cache
from kernel_ops import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


@pytest.mark.parametrize("group", [1, 2, 17])
@pytest.mark.parametrize("requests,kv_heads", [(1, 8), (7, 9), (8, 8)])
@pytest.mark.parametrize("longest", [1, 640, 641, 1024, 1025])
def test_against_64_bits(group, requests, kv_heads, longest):
    ops, D, heads = HipOps(), 64, group * kv_heads
    lengths = [max(1, longest - 61 * i) for i in range(requests)]         # keys, the step's own among them
    cache = make_cache(kv_heads, D, 2, BF, n_pages=sum((n + 15) // 16 for n in lengths), slots=requests, max_context=longest)
    g = torch.Generator().manual_seed(longest + requests)
    kv = cache.layer_cache(1).kv
    kv.k.copy_(torch.randn(kv.k.shape, generator=g).to(BF))
    kv.v.copy_(torch.randn(kv.v.shape, generator=g).to(BF))
    slots = [cache.open() for _ in lengths]
    for slot, n in zip(slots, lengths):
        assert cache.prepare(slot, 0, n)
    batch, keep = build_batch(ops, cache, [SimpleNamespace(slot=s, start_pos=n - 1, tokens=[0], want=[0]) for s, n in zip(slots, lengths)])
    q, k, v = (torch.randn(requests, w, generator=g).to(BF).to(DEV) for w in (heads * D, kv_heads * D, kv_heads * D))
    outs = []
    for bound in (0, longest, 4096):       # as it is, as a recorded step sees it, and sized for more
        batch.context_bound = bound
        out = torch.zeros(requests, heads * D, dtype=BF, device=DEV)
        ops.attention_decode_fresh(q, k, v, out, None, None, 1e-6, None, heads, kv_heads, D, D ** -0.5, None, batch, kv)
        outs.append(out)
    # (the step wrote its keys and values into the pages)
    table, K, V = kv.table.cpu(), kv.k[:, 1].double().cpu(), kv.v[:, 1].double().cpu()
    for i, n in enumerate(lengths):
        pages = table[slots[i], :(n + 15) // 16].long()
        keys = K[pages].permute(1, 0, 2, 3).reshape(kv_heads, -1, D)[:, :n]
        values = V[pages].permute(1, 0, 3, 2).reshape(kv_heads, -1, D)[:, :n]
        assert torch.equal(keys[:, -1].reshape(-1), k[i].double().cpu()) and torch.equal(values[:, -1].reshape(-1), v[i].double().cpu())
        p = torch.softmax(q[i].double().cpu().view(kv_heads, group, D) @ keys.transpose(1, 2) * D ** -0.5, -1)
        want = (p @ values).reshape(-1)
        # weights and result are rounded to bfloat16: 2^-9 of the values' weighted sizes each, and the 32-bit scores
        bound = ((p @ values.abs()).reshape(-1) + want.abs()) * 2.0 ** -9 * 1.05 + 1e-5
        for out in outs:
            assert bool(((out[i].double().cpu() - want).abs() <= bound).all())
