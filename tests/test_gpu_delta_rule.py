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


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("at", [0, 15, 100, 127, 129, 199])
def test_a_value_that_is_not_finite_reaches_no_earlier_token(value, at):
    """One value of one token: the outputs before it are what they are without it, those from it on are not finite."""
    case, H, V, column = Portions([200], 2, 4, 64, "apart", 0.05, 0.3), 4, 64, 70
    clean = case.run(True)[0]
    case.v[at, column] = value
    out = case.run(True)[0]
    assert torch.equal(out[:at], clean[:at])
    assert not bool(torch.isfinite(out[at:, column]).any())
    others = [c for c in range(H * V) if c != column]
    assert torch.equal(out[:, others], clean[:, others])


# (sizes with two, four and eight wavefronts a head and with 8 and 16 rows of S each)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("G,H,D,V,mean,pace", [(8, 16, 64, 64, 0.0, 0.0), (4, 8, 64, 64, 1.0, -3.0), (2, 8, 64, 32, 0.5, -1.0),
                                               (2, 16, 32, 64, 0.5, -3.0), (4, 4, 128, 64, 1.0, -2.0)])
def test_a_step_in_one_kernel_is_no_further_from_the_exact_result_than_in_four(G, H, D, V, mean, pace, dtype):
    """60 steps of three requests, in one kernel and in four, each from the state that it left itself; the exact
    ones from the convolved, normed inputs that both make alike.  (bfloat16: the rounding of the result is nearly all of
    the distance in both.)"""
    n, taps, steps, eps = 3, 4, 60, 1e-6
    C = 2 * G * D + H * V
    ld, col_b, col_a = C + H * V + 2 * H, C + H * V, C + H * V + H
    gen = torch.Generator().manual_seed(5)
    rand = lambda *shape: torch.randn(*shape, generator=gen).to(DEV)
    conv_w, a_log, dt_bias, norm_w = 0.5 * rand(C, taps) + 0.3 * mean, pace + 0.5 * rand(H), rand(H), 1.0 + 0.1 * rand(V)
    saved = [(rand(n, taps - 1, C) + mean)] * 2
    states = [0.3 * rand(n, H, D, V)] * 2
    saved, states = [t.clone() for t in saved], [t.clone() for t in states]
    exact = states[0].double()
    slots, cu, seq, zero = ints([2, 0, 1]), ints([0, 1, 2, 3]), ints([0, 1, 2]), ints([0, 0, 0])
    conv_stride, stride = ctypes.c_size_t((taps - 1) * C), ctypes.c_size_t(H * D * V)
    lib, code = native.lib(), int(dtype == torch.bfloat16)
    qk, v, gates, o = (torch.empty(n, w, device=DEV) for w in (2 * G * D, H * V, 2 * H, H * V))
    off, size = [0.0, 0.0], 0.0
    for _ in range(steps):
        proj, outs = (rand(n, ld) + mean).to(dtype), [torch.empty(n, H * V, dtype=dtype, device=DEV) for _ in range(2)]
        gate = ctypes.c_void_p(proj.data_ptr() + proj.element_size() * C)
        check(lib.celeg_delta_prepare(ptr(proj), ld, code, col_b, col_a, ptr(conv_w), ptr(a_log), ptr(dt_bias), ptr(saved[0]), conv_stride,
                                      ptr(zero), ptr(seq), ptr(zero), ptr(slots), ptr(qk), ptr(v), ptr(gates), n, G, H, D, V, taps, None))
        check(lib.celeg_delta_conv_state(ptr(proj), ld, code, ptr(saved[0]), conv_stride, ptr(cu), ptr(slots), n, C, taps, None))
        check(lib.celeg_delta_scan(ptr(qk), ptr(v), ptr(gates), ptr(states[0]), stride, ptr(cu), ptr(slots), ptr(o), n, G, H, D, V, 0, ptr(seq),
                                   None, n, NO_LIMIT, None))
        check(lib.celeg_delta_gated_norm(ptr(o), ptr(norm_w), gate, ld, code, ctypes.c_float(eps), ptr(outs[0]), n, H, V, 0, None))
        check(lib.celeg_delta_step(ptr(proj), ld, code, col_b, col_a, ptr(conv_w), ptr(a_log), ptr(dt_bias), ptr(saved[1]), conv_stride,
                                   ptr(states[1]), stride, ptr(slots), ptr(norm_w), gate, ld, ctypes.c_float(eps), 0, ptr(outs[1]), n, G, H, D,
                                   V, taps, None))
        heads = qk.double().view(n, 2, G, D).repeat_interleave(H // G, 2)
        z = proj[:, C:C + H * V].double().view(n, H, V)
        for t in range(n):
            row, slot = slice(t, t + 1), int(slots[t])
            y, exact[slot] = recurrence(heads[row, 0], heads[row, 1], v[row].double().view(1, H, V), gates[row, :H].double(),
                                        gates[row, H:].double(), exact[slot])
            y = y[0] / torch.sqrt((y[0] ** 2).mean(-1, keepdim=True) + eps) * norm_w.double() * torch.nn.functional.silu(z[t])
            size += float((y ** 2).sum())
            for i in range(2):
                off[i] += float(((outs[i][t].double().view(H, V) - y) ** 2).sum())
        assert torch.equal(saved[0], saved[1])
    assert math.sqrt(off[1] / size) <= (1.0 if dtype == torch.float32 else 1.01) * math.sqrt(off[0] / size)
    # (both round the state once a step in the same way; what differs, the sums that go into it, is the smaller part)
    assert distance(states[1], exact) <= 1.02 * distance(states[0], exact)
