"""Few tokens of the two recurrences (scan_kernel): rows of the state in quads, and one by one where sizes or addresses do not allow
quads, against float64.

Tolerance: all arithmetic is float32 on the operands given; a sum over `dim` products has a relative error of at most (dim / 16 + 4) 2^-24 of
its absolute sum, decays and exponentials 2^-22: 1e-5 of the largest value covers 256 rows with room for cancellation."""
import pytest
import torch

from polarquant_amd import recurrent_ops as ops
from polarquant_amd.recurrent_ops import Step

pytestmark = pytest.mark.gpu


def shifted(t):
    """The same values one element past an allocation's start."""
    return torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)


def off(got, want):
    return float((got.double() - want).abs().max() / want.abs().max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("dim,vdim,H,G,L,aligned", [(128, 128, 4, 2, 1, True), (128, 128, 4, 4, 1, False), (4, 16, 2, 1, 3, True), (60, 33, 3, 3, 2, True),
                                                    (64, 48, 2, 2, 16, True), (132, 20, 2, 1, 5, True), (256, 64, 1, 1, 4, True), (30, 17, 2, 2, 3, True)])
def test_delta(dim, vdim, H, G, L, aligned, dtype):
    g = torch.Generator(device="cuda").manual_seed(dim + L)
    B, r = 2, lambda *s: torch.randn(*s, generator=g, device="cuda")
    q, k, v = r(B * L, G * dim).to(dtype), r(B * L, G * dim).to(dtype), r(B * L, H * vdim).to(dtype)
    q_inv, k_inv, log_g, beta = r(B * L, G).abs() * 0.1, r(B * L, G).abs() * 0.1, -r(B * L, H * dim).abs(), torch.sigmoid(r(B * L, H))
    S0 = r(B, H, vdim, dim)
    state = S0.clone()
    o = ops.delta_scan(ops.DeltaInputs(*[t if aligned else shifted(t) for t in (q, k)], v, q_inv, k_inv, log_g, beta), state, Step(B, L, 7))
    S, per = S0.double(), H // G
    heads = lambda t, n, d: t.double().view(B, L, n, d)
    kq = [(heads(t, G, dim) * i.double().view(B, L, G, 1)).repeat_interleave(per, 2) for t, i in ((k, k_inv), (q, q_inv))]
    want = []
    for t in range(L):
        S = S * heads(log_g, H, dim)[:, t].exp()[:, :, None]
        u = beta.double().view(B, L, H, 1)[:, t] * (heads(v, H, vdim)[:, t] - (S * kq[0][:, t, :, None]).sum(-1))
        S = S + u[..., None] * kq[0][:, t, :, None]
        want.append((S * kq[1][:, t, :, None]).sum(-1))
    assert off(state, S) < 1e-5 and off(o, torch.stack(want, 1).reshape(B * L, H * vdim)) < 1e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("dim,vdim,H,L,pad", [(128, 256, 2, 1, 0), (128, 256, 2, 1, 1), (8, 15, 3, 3, 0), (100, 40, 2, 2, 0), (192, 16, 1, 7, 4), (34, 8, 2, 2, 0)])
def test_memory(dim, vdim, H, L, pad, dtype):
    g = torch.Generator(device="cuda").manual_seed(dim + L)
    B, r = 2, lambda *s: torch.randn(*s, generator=g, device="cuda")
    p = r(B * L, 2 * H * dim + H * vdim + pad).to(dtype)                    # (pad: rows that are no multiple of four elements apart)
    q, k, v = p[:, :H * dim], p[:, H * dim:2 * H * dim], p[:, 2 * H * dim:2 * H * dim + H * vdim]
    log_i, log_f = r(B * L, H), -r(B * L, H).abs()
    state, m = ops.memory_state(B, H, dim, vdim, "cuda")
    state.copy_(r(*state.shape))
    S0 = state.double()
    o, den = ops.memory_scan(q, k, v, log_i, log_f, state, m, 0.3, Step(B, L, 7))
    heads = lambda t, d: t.double().reshape(B, L, H, d)
    S, mx, want, wden = S0, torch.zeros(B, H, dtype=torch.float64, device="cuda"), [], []
    v1 = torch.cat([heads(v, vdim), torch.ones(B, L, H, 1, dtype=torch.float64, device="cuda")], -1)
    for t in range(L):
        i, f = log_i.double().view(B, L, H)[:, t], log_f.double().view(B, L, H)[:, t]
        new = torch.maximum(f + mx, i)
        S = (f + mx - new).exp()[..., None, None] * S + (i - new).exp()[..., None, None] * v1[:, t, :, :, None] * heads(k, dim)[:, t, :, None]
        mx = new
        e = (S * heads(q, dim)[:, t, :, None]).sum(-1) * 0.3
        want.append(e[..., :-1])
        wden.append(torch.maximum(e[..., -1].abs(), (-mx).exp()) + 1e-6)
    assert off(state, S) < 1e-5 and off(m[:, :, 0], mx) < 1e-5
    assert off(o, torch.stack(want, 1).reshape(B * L, H * vdim)) < 1e-5 and off(den, torch.stack(wden, 1).reshape(B * L, H)) < 1e-5


@pytest.mark.parametrize("dim", [100, 30])                                  # (quads with rows to spare; row by row)
def test_infinite_state(dim):
    """An infinite entry of the state makes its column's result infinite where q does not vanish, and nothing NaN: no other row repeats it."""
    B, H, vdim = 1, 1, 20
    g = torch.Generator(device="cuda").manual_seed(dim)
    q, k, v = torch.randn(B, 2 * dim + vdim, generator=g, device="cuda").split((dim, dim, vdim), 1)
    log_i, log_f = torch.full((B, H), -1.0, device="cuda"), torch.full((B, H), -0.5, device="cuda")
    state, m = ops.memory_state(B, H, dim, vdim, "cuda")
    state[:, :, 7, 1], q[:, 1] = float("inf"), -2.0
    o, _ = ops.memory_scan(q, k, v, log_i, log_f, state, m, 0.3, Step(B, 1, 7))
    assert float(o[0, 7]) == float("-inf") and int(torch.isinf(state).sum()) == 1 and not torch.isnan(state).any()
    assert bool(torch.isfinite(o).sum() == vdim - 1)
