"""The gated delta rule's kernels by themselves, called as the host code calls them, against the recurrence in 64 bits:
a form that takes the chain of tokens' place may not be further from the exact result than the chain is."""
import ctypes
import math

import pytest
import torch

from celeg_amd import native

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NO_LIMIT = 2 ** 31 - 1


def check(code):
    assert code == 0, f"error {code}"


def ptr(t):
    return ctypes.c_void_p(t.data_ptr() if t is not None else None)


def ints(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def unit_rows(shape, kind, gen):
    """Unit vectors: independent, all alike, or of four dimensions."""
    n = shape[-1]
    if kind == "few":
        x = torch.randn(*shape[:-1], 4, generator=gen, dtype=torch.float64) @ torch.randn(4, n, generator=gen, dtype=torch.float64)
    else:
        x = torch.randn(*shape, generator=gen, dtype=torch.float64) + (1.0 if kind == "alike" else 0.0)
    return x / x.norm(dim=-1, keepdim=True)


def recurrence(q, k, v, beta, decay, state):
    """q, k [T, H, D], v [T, H, V], beta, decay [T, H], state [H, D, V], all 64-bit -> (outputs [T, H, V], state)"""
    S, out = state.clone(), torch.empty_like(v)
    for t in range(q.shape[0]):
        S = S * decay[t, :, None, None]
        u = beta[t, :, None] * (v[t] - (k[t, :, :, None] * S).sum(1))
        S = S + k[t, :, :, None] * u[:, None, :]
        out[t] = (q[t, :, :, None] * S).sum(1)
    return out, S


def distance(got, want):
    return float((got.double() - want).norm() / want.norm())


class Portions:
    """Rows of several requests' portions: what delta_prepare leaves, and the states before them."""

    def __init__(self, lens, G, H, V, kind, pace, start, seed=3):
        gen = torch.Generator().manual_seed(seed)
        D, T, n = 64, sum(lens), len(lens)
        self.sizes, self.lens = (G, H, D, V), lens
        q, k = unit_rows((T, G, D), kind, gen) / math.sqrt(D), unit_rows((T, G, D), kind, gen)
        z = torch.randn(2, T, H, generator=gen, dtype=torch.float64)
        beta = torch.sigmoid(z[0])
        decay = torch.exp(-pace * torch.exp(z[1]) * torch.nn.functional.softplus(torch.randn(T, H, generator=gen, dtype=torch.float64)))
        self.qk = torch.cat([q, k], 1).reshape(T, 2 * G * D).float().to(DEV)
        self.v = torch.randn(T, H * V, generator=gen).to(DEV)
        self.gates = torch.cat([beta, decay], 1).float().to(DEV)
        self.states = (start * torch.randn(n, H, D, V, generator=gen)).to(DEV)
        self.cu = ints([sum(lens[:i]) for i in range(n + 1)])
        self.slots = ints(list(reversed(range(n))))
        self.seq = ints([i for i, m in enumerate(lens) for _ in range(m)])

    def exact(self):
        G, H, D, V = self.sizes
        T = self.qk.shape[0]
        qk = self.qk.double().view(T, 2, G, D).repeat_interleave(H // G, 2)
        outs, states = [], self.states.double().clone()
        for i, m in enumerate(self.lens):
            rows = slice(sum(self.lens[:i]), sum(self.lens[:i]) + m)
            slot = len(self.lens) - 1 - i
            o, states[slot] = recurrence(qk[rows, 0], qk[rows, 1], self.v[rows].double().view(m, H, V), self.gates[rows, :H].double(),
                                         self.gates[rows, H:].double(), states[slot])
            outs.append(o)
        return torch.cat(outs).view(T, H * V), states

    def run(self, chunks):
        G, H, D, V = self.sizes
        lib, T, n = native.lib(), self.qk.shape[0], len(self.lens)
        out, states = torch.full_like(self.v, float("nan")), self.states.clone()
        stride = ctypes.c_size_t(H * D * V)
        if chunks:
            count = sum((m + 63) // 64 for m in self.lens)
            lib.celeg_delta_chunks_floats.restype = ctypes.c_longlong
            ws = torch.empty(lib.celeg_delta_chunks_floats(count, H, V), device=DEV)
            check(lib.celeg_delta_chunks(ptr(self.qk), ptr(self.v), ptr(self.gates), ptr(states), stride, ptr(self.cu), ptr(self.slots), ptr(out),
                                         ptr(ws), n, count, 1, G, H, D, V, None))
        else:
            pairs = torch.empty(T, 4 * G, device=DEV)
            check(lib.celeg_delta_scan(ptr(self.qk), ptr(self.v), ptr(self.gates), ptr(states), stride, ptr(self.cu), ptr(self.slots), ptr(out),
                                       n, G, H, D, V, 0, ptr(self.seq), ptr(pairs), T, NO_LIMIT, None))
        torch.cuda.synchronize()
        return out, states


# (pace: no decay, decays near one, ordinary and strong ones; start: the size of the states before)
@pytest.mark.parametrize("lens,G,H,V,kind,pace,start", [
    ([256], 2, 4, 64, "apart", 1.0, 0.0), ([320], 2, 4, 64, "alike", 0.05, 0.0), ([192, 65], 2, 2, 16, "alike", 0.0, 0.3),
    ([300], 1, 2, 128, "few", 0.05, 0.3), ([256], 4, 4, 48, "few", 0.0, 0.3), ([1, 191, 64], 2, 4, 64, "apart", 8.0, 0.3),
    ([448], 2, 4, 64, "alike", 1.0, 0.3)])
def test_chunks_are_no_further_from_the_exact_result_than_the_chain(lens, G, H, V, kind, pace, start):
    case = Portions(lens, G, H, V, kind, pace, start)
    want, want_states = case.exact()
    (out, states), (chain_out, chain_states) = case.run(True), case.run(False)
    assert distance(out, want) <= distance(chain_out, want)
    assert distance(states, want_states) <= distance(chain_states, want_states)
