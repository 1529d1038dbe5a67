"""Causal attention of a prompt (prompt_attn_kernel) against float64, at the edges of its tiles (128 queries, 64 keys, 16-byte pieces of
a row).

Tolerance: weights and result are rounded to the dtype, each by at most half a unit in the last place u (2^-8 bf16, 2^-11 fp16); the
errors of a row's weights are independent, so the relative 2-norm error stays below u."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
UNIT = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def reference(q, k, v, scale, start=None, sink=None):
    """q [B, L, H, D], k [B, Lk, G, D], v [B, Lk, G, Dv] -> [B, L, H, Dv]; the queries are the last of the keys' tokens."""
    (B, L, H, _), (Lk, G) = q.shape, k.shape[1:3]
    q, k, v = [t.double().transpose(1, 2) for t in (q, k, v)]
    k, v = k.repeat_interleave(H // G, 1), v.repeat_interleave(H // G, 1)
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) * scale
    i, j = torch.arange(L, device=q.device)[:, None] + (Lk - L), torch.arange(Lk, device=q.device)
    hidden = (j > i)[None, None].expand(B, 1, L, Lk)
    if start is not None:
        hidden = hidden | (j < start[:, None, None, None])
    s = s.masked_fill(hidden, -math.inf)
    if sink is not None:
        s = torch.cat([s, sink.double()[None, :, None, None].expand(B, H, L, 1)], -1)
    return torch.matmul(s.softmax(-1)[..., :Lk], v).transpose(1, 2)


def off(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,L,Lk,H,D,Dv,scale", [
    (1, 1, 1, 1, 128, 128, 0.1), (2, 63, 63, 8, 128, 128, 0.09), (1, 64, 64, 3, 64, 64, 0.2), (1, 65, 65, 8, 128, 128, -0.09), (1, 127, 255, 2, 128, 128, 0.0),
    (1, 129, 129, 16, 128, 128, 1.0), (2, 200, 333, 5, 72, 40, 0.1), (1, 257, 257, 2, 192, 128, 0.07), (1, 130, 449, 2, 256, 256, 0.06)])
def test_values_by_channel(B, L, Lk, H, D, Dv, scale, dtype):
    from polarquant_amd.latent_ops import latent_prefill_attention
    g = torch.Generator(device="cuda").manual_seed(L + Lk)
    q, k, v = [torch.randn(B, n, H, d, generator=g, device="cuda").to(dtype) for n, d in ((L, D), (Lk, D), (Lk, Dv))]
    sink = torch.randn(H, generator=g, device="cuda")
    start = torch.tensor([0] * (B - 1) + [(Lk - L) // 2], dtype=torch.int32, device="cuda")
    vt = torch.zeros(B, H, Dv, -(-Lk // 64) * 64, dtype=dtype, device="cuda")
    vt[..., :Lk] = v.permute(0, 2, 3, 1)
    got = latent_prefill_attention(q, k, vt, sink, scale, None, start).view(B, L, H, Dv)
    assert off(got, reference(q, k, v, scale, start, sink)) < UNIT[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,L,N,Nk,layout", [(1, 1, 4, 4, "tokens"), (2, 63, 8, 2, "heads"), (1, 64, 7, 1, "tokens"), (3, 65, 28, 4, "slices"),
                                             (1, 128, 32, 8, "slices"), (2, 129, 5, 5, "expanded"), (1, 515, 16, 8, "tokens")])
def test_values_by_token(B, L, N, Nk, layout, dtype):
    """The strides that callers have: transposed views of [B, L, heads, 128], contiguous heads, slices of one projection, a batch that
    is one expanded sequence."""
    from polarquant_amd.attention import prompt_attention, prompt_attention_takes
    g = torch.Generator(device="cuda").manual_seed(7 * L)
    if layout == "slices":
        p = torch.randn(B, L, N + 2 * Nk, 128, generator=g, device="cuda").to(dtype).transpose(1, 2)
        q, k, v = p[:, :N], p[:, N:N + Nk], p[:, N + Nk:]
    else:
        q, k, v = [torch.randn(1 if layout == "expanded" else B, L, n, 128, generator=g, device="cuda").to(dtype).transpose(1, 2) for n in (N, Nk, Nk)]
        if layout == "heads":
            q, k, v = [t.contiguous() for t in (q, k, v)]
        if layout == "expanded":
            q, k, v = [t.expand(B, -1, -1, -1) for t in (q, k, v)]
    assert prompt_attention_takes(q, k, v)
    got = prompt_attention(q, k, v)
    assert got.shape == (B, L, N, 128) and off(got, reference(*[t.transpose(1, 2) for t in (q, k, v)], 128 ** -0.5)) < UNIT[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("form", ["channel", "token", "window"])
def test_the_largest_weight_is_exact(form, dtype):
    """A key of the first tile, then one of the second that exceeds it by 0.2 to 5 and is the only one with values.  Its weight is 1 in any
    dtype, so that what is left is the rounding of the result: the nearest number, but for the float32 sums' 1e-6 of a unit that is
    2^-8 or 2^-11.  A weight that is itself rounded moves about a quarter of the results to a neighbour."""
    from polarquant_amd import recurrent_ops
    from polarquant_amd.attention import prompt_attention
    from polarquant_amd.latent_ops import latent_prefill_attention
    g = torch.Generator(device="cuda").manual_seed(3)
    L, H = 130, 24
    q, k, v = [torch.zeros(1, L, H, 128, device="cuda", dtype=dtype) for _ in range(3)]
    q[..., 0] = 1.0
    k[..., 0] = -40.0
    k[:, 3, :, 0] = 0.0
    k[:, 100, :, 0] = torch.linspace(0.2, 5.0, H, device="cuda").to(dtype)
    v[:, 100] = torch.randn(1, H, 128, generator=g, device="cuda").to(dtype)
    if form == "channel":
        sink, vt = torch.full((H,), -60.0, device="cuda"), torch.zeros(1, H, 128, 192, device="cuda", dtype=dtype)
        vt[..., :L] = v.permute(0, 2, 3, 1)
        got = latent_prefill_attention(q, k, vt, sink, 1.0).view(1, L, H, 128)
    elif form == "token":
        got = prompt_attention(*[t.transpose(1, 2) for t in (q, k, v)], 1.0)
    else:
        ring, out = recurrent_ops.WindowRing(1, H, 128, 128, L, dtype, "cuda"), torch.empty(L, H * 128, device="cuda", dtype=dtype)
        got = recurrent_ops.window_attention(q.view(L, -1), ring, None, 1.0, recurrent_ops.Step(1, L, 0), out, 1.0, k.view(L, -1), v.view(L, -1)).view(1, L, H, 128)
    want = reference(q, k, v, 1.0)[:, 100:].to(dtype)
    assert float((got[:, 100:] != want).float().mean()) < 0.005


def test_what_prompt_attention_refuses():
    from polarquant_amd.attention import prompt_attention_takes
    x = torch.randn(2, 4, 70, 128, device="cuda").bfloat16()
    assert prompt_attention_takes(x, x[:, :2], x[:, :2])
    assert not prompt_attention_takes(x, x[:, :3], x[:, :3])                       # heads that do not share evenly
    assert not prompt_attention_takes(x.float(), x.float(), x.float())
    assert not prompt_attention_takes(x[..., :64], x[..., :64], x[..., :64])
    y = torch.randn(2 * 4 * 70 * 132, device="cuda").bfloat16().view(2, 4, 70, 132)
    assert not prompt_attention_takes(y[..., :128], x, x)                          # rows 132 apart
    z = torch.randn(2 * 4 * 70 * 128 + 4, device="cuda").bfloat16()[4:].view(2, 4, 70, 128)
    assert not prompt_attention_takes(z, x, x)                                     # 8-byte aligned
    # what the grid or the C ABI do not hold: the caller falls back instead of meeting an error
    w = x[:1, :1, :1]
    for B, N, L in ((65536, 1, 1), (1, 65536, 1), (1, 1, 65535 * 128 + 1), (1, 0, 1), (0, 1, 1)):
        wide = w.expand(B, N, L, 128) if B and N else x.new_empty(B, N, L, 128)
        assert not prompt_attention_takes(wide, wide, wide)
    assert prompt_attention_takes(*[w.expand(1, 1, 65535 * 128, 128)] * 3) and not prompt_attention_takes(x, x[:, :0], x[:, :0]) and not prompt_attention_takes(x[0], x[0], x[0])


def test_a_prompt_of_one_token_is_the_librarys(monkeypatch):
    """Its attention is a copy of the values; the library needs 6 us for it, whatever the batch, a tile of the kernel 7 to 14."""
    from polarquant_amd import modeling_common as mc
    taken, own = [], mc.prompt_attention
    monkeypatch.setattr(mc, "prompt_attention", lambda q, k, v: (taken.append(q.shape[2]), own(q, k, v))[1])
    with torch.no_grad():
        for L in (1, 2, 3):
            q, k, v = [torch.randn(2, n, L, 128, device="cuda").bfloat16() for n in (8, 2, 2)]
            got = mc._prefill_attention(q, k, v, None, 4, True)
            assert got.shape == (2, L, 8, 128) and off(got, reference(*[t.transpose(1, 2) for t in (q, k, v)], 128 ** -0.5)) < UNIT[torch.bfloat16]
    assert taken == [2, 3]
