"""What this framework is timed on: the calls its users make, as plain cases.

`listed()` has the fixed cases, `draw(rng)` one more of the same ranges.  `prepare` makes what a program has in hand before the
call (on the GPU, from the seed alone), `run` is one pass through public entry points, `work` what a pass cannot do without,
`exact` the same result in 64 bits from plain torch, `tolerance` how far a correct implementation may be from another.

Operations ("op"):
  scores  scores of one query against a quantized key cache (`attention_decode_forward_triton_impl`)
  attend  one step of decode attention over a polar key cache, values in 16 or 4 bits (`polar_decode_attention`, `.._v4`)
  append  quantization of a prompt's keys, and with 4-bit values of its values (`quantize_and_pack_nbit`, `quantize_values`)
  prompt  a prompt and the first token after it through a model of one of the three families (`model(...)`)
  decode  one token of running sequences, replayed from the model's captured step (`model.graph_decoder`)
"""
import math

import torch

GROUP, PAIRS, DIM = 128, 64, 128
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}
VOCAB = 32768
STEPS = 8192                            # tokens a decoded sequence may grow by

# Widths of the models: those the package's own benchmarks compare its families at, two layers of each.
SIZES = {"large": dict(width=4096, heads=32, kv_heads=8, ff=14336, q_rank=1536, kv_rank=512, window=2048, memory_heads=16, rank=128),
         "medium": dict(width=2048, heads=16, kv_heads=8, ff=8192, q_rank=768, kv_rank=256, window=1024, memory_heads=8, rank=64)}
LAYERS = 2
HEADS = [(32, 8), (32, 32), (28, 4), (16, 8)]       # query and KV heads
BITS = [(4, 4), (4, 4), (3, 3), (4, 3)]             # radius and angle


def listed():
    return [
        # the reference's own micro-benchmark call: multi-head, 4k context; 9 MB, so launch and latency
        dict(name="scores_mha_4k", op="scores", batch=1, heads=32, kv_heads=32, tokens=4096, rbits=4, tbits=4, dtype="float16"),
        # a chat turn: one sequence, short context, 7 query heads per KV head
        dict(name="attend_b1_2k", op="attend", batch=1, heads=28, kv_heads=4, tokens=2000, rbits=4, tbits=4, dtype="bfloat16", values=16,
             ragged=False, padded=False),
        # the headline: a served batch at long context
        dict(name="attend_b16_32k", op="attend", batch=16, heads=32, kv_heads=8, tokens=32769, rbits=4, tbits=4, dtype="float16", values=16,
             ragged=False, padded=False),
        # continuous batching: sequences of 512 to 8192 tokens, 3-bit codes
        dict(name="attend_ragged_b64", op="attend", batch=64, heads=28, kv_heads=4, tokens=8192, rbits=3, tbits=3, dtype="float16", values=16,
             ragged=True, padded=False),
        # the Mixed variant: values in 4 bits as well
        dict(name="attend_values4_b8_16k", op="attend", batch=8, heads=32, kv_heads=8, tokens=16421, rbits=4, tbits=4, dtype="bfloat16", values=4,
             ragged=False, padded=False),
        # a long prompt's keys go to the cache
        dict(name="append_b1_128k", op="append", batch=1, kv_heads=8, tokens=131072, rbits=4, tbits=4, dtype="float16", values=16, eager_gpu=False),
        # time to the first tokens, in each family
        dict(name="prompt_polar_8k", op="prompt", family="polar", size="large", batch=1, tokens=8192, values=16),
        dict(name="prompt_latent_8k", op="prompt", family="latent", size="large", batch=1, tokens=8192, values=16),
        dict(name="prompt_recurrent_8k", op="prompt", family="recurrent", size="large", batch=1, tokens=8192, values=16),
        # a token of a served batch, in each family
        dict(name="decode_polar_b8_4k", op="decode", family="polar", size="large", batch=8, tokens=4096, values=16),
        dict(name="decode_latent_b8_4k", op="decode", family="latent", size="large", batch=8, tokens=4096, values=16),
        dict(name="decode_recurrent_b8_2k", op="decode", family="recurrent", size="large", batch=8, tokens=2048, values=16),
    ]


def draw(rng):
    def spread(lo, hi):                 # even over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["attend", "attend", "attend", "append", "append", "scores", "prompt", "prompt", "decode", "decode"])
    rbits, tbits = rng.choice(BITS)
    dtype = rng.choice(sorted(DTYPES))
    if op in ("prompt", "decode"):
        family, size = rng.choice(["polar", "latent", "recurrent"]), rng.choice(sorted(SIZES))
        values = rng.choice([16, 16, 4]) if family == "polar" else 16
        tokens = spread(48, 8192)
        batch = spread(1, max(1, min(8, 8192 // tokens))) if op == "prompt" else spread(1, 8 if tokens <= 4096 else 4)
        return dict(op=op, family=family, size=size, batch=batch, tokens=tokens, values=values)
    heads, kv_heads = rng.choice(HEADS)
    most = 16 * 8 * 32768               # cached tokens times KV heads, the listed largest
    if op == "scores":
        batch = spread(1, 8)
        return dict(op=op, batch=batch, heads=heads, kv_heads=kv_heads, tokens=GROUP * spread(1, min(256, most // (batch * kv_heads * GROUP))),
                    rbits=rbits, tbits=tbits, dtype=dtype)
    if op == "append":
        batch = spread(1, 16)
        return dict(op=op, batch=batch, kv_heads=kv_heads, tokens=GROUP * spread(1, min(1024, 1048576 // (batch * kv_heads * GROUP))), rbits=rbits,
                    tbits=tbits, dtype=dtype, values=rng.choice([16, 4]), eager_gpu=rng.random() < 0.5)
    batch = spread(1, 64)
    values = rng.choice([16, 16, 4])
    kind = rng.random()
    return dict(op=op, batch=batch, heads=heads, kv_heads=kv_heads, tokens=spread(64, min(131072, most // (batch * kv_heads))), rbits=rbits, tbits=tbits,
                dtype=dtype, values=values, ragged=batch > 1 and values == 16 and kind < 0.35, padded=batch > 1 and kind > 0.8)


# ----------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, dtype):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _rotate(x, cos, sin):
    a, b = x[..., :PAIRS], x[..., PAIRS:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _angles(tokens, theta, dtype=torch.float32, first=0):
    f = 1.0 / theta ** (torch.arange(0, DIM, 2, device="cuda", dtype=torch.float32) / DIM)
    return torch.arange(first, first + tokens, device="cuda", dtype=dtype)[:, None] * f.to(dtype)


def _keys(g, heads, tokens, dtype):
    """[heads, tokens, 128] as a model leaves them: normal, 4 channels 8 times as large, rotated by position."""
    k = torch.randn(heads, tokens, DIM, generator=g, device="cuda")
    k[..., torch.randperm(DIM, generator=g, device="cuda")[:4]] *= 8.0
    a = _angles(tokens, 5e5)
    return _rotate(k, a.cos(), a.sin()).to(dtype)


def _quantize(k, rbits, tbits, dtype):
    """k [.., groups * 128, 128] -> codes and the four group constants; the decode operations take any such codes."""
    x = k.float().unflatten(-2, (-1, GROUP)).unflatten(-1, (2, PAIRS))
    phi = torch.atan2(x[..., 1, :], x[..., 0, :])
    phi, r = torch.where(phi < 0, phi + 2 * math.pi, phi), x.square().sum(-2).sqrt()

    def bins(v, bits):
        lo, hi = v.amin(-2, keepdim=True), v.amax(-2, keepdim=True)
        step = (hi - lo) / 2 ** bits
        return ((v - lo) / step).floor().clamp_(0, 2 ** bits - 1).to(torch.uint8), step.to(dtype), lo.to(dtype)

    theta, tscale, tmn = bins(phi, tbits)
    rho, rscale, rmn = bins(r, rbits)
    return (rho << tbits) + theta, rscale, rmn, tscale, tmn


def _quantize_values(v, dtype):
    """v [.., tokens, 128] -> 4-bit codes, eight to an int32, scale and zero point of each row."""
    x = v.float()
    lo, hi = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    scale, lo = ((hi - lo) / 15).to(dtype), lo.to(dtype)
    q = ((x - lo.float()) / scale.float()).round().clamp_(0, 15).to(torch.int64).unflatten(-1, (16, 8))
    word = (q << torch.arange(0, 32, 4, device=v.device)).sum(-1)
    return torch.where(word >= 1 << 31, word - (1 << 32), word).to(torch.int32), scale, lo


def _prepare_cache(c, seed):
    g, dt = _generator(seed), DTYPES[c["dtype"]]
    B, N, Nk, T = c["batch"], c["heads"], c["kv_heads"], c["tokens"]
    s = {"q": _normal(g, B, N, 1, DIM, dtype=dt)}
    if c["op"] == "scores":
        parts = [_quantize(_keys(g, Nk, T, dt), c["rbits"], c["tbits"], dt) for _ in range(B)]
        return dict(s, cache=[torch.stack(t) for t in zip(*parts)])
    if c["ragged"]:                     # lengths from a sixteenth of the longest on
        lengths = torch.randint(max(1, T // 16), T + 1, (B,), generator=torch.Generator().manual_seed(seed))
        T = int(lengths.max())
    else:
        lengths = torch.full((B,), T)
    groups = (T - 1) // GROUP           # the newest key is always in the window of unquantized ones
    per_seq = (lengths - 1) // GROUP
    parts, window, values, v4 = [], torch.zeros(B, Nk, GROUP, DIM, dtype=dt, device="cuda"), [], []
    for b in range(B):
        k = _keys(g, Nk, groups * GROUP + GROUP, dt)
        if groups:
            parts.append(_quantize(k[:, :groups * GROUP], c["rbits"], c["tbits"], dt))
        n = int(lengths[b] - per_seq[b] * GROUP)
        window[b, :, :n] = k[:, groups * GROUP:groups * GROUP + n]
        v = _normal(g, Nk, groups * GROUP + GROUP, DIM, dtype=dt)
        if c["values"] == 4:
            if groups:
                v4.append(_quantize_values(v[:, :groups * GROUP], dt))
            v = v[:, groups * GROUP:]
        values.append(v)
    s.update(cache=[torch.stack(t) for t in zip(*parts)] if groups else [None] * 5, window=window, v=torch.stack(values), groups=groups,
             resid=int(T - groups * GROUP), mask=None, per_seq=None, resid_per_seq=None, total=None,
             v4=([torch.stack(t) for t in zip(*v4)] if groups else [None] * 3) if c["values"] == 4 else None)
    if c["ragged"]:
        s.update(per_seq=per_seq.to("cuda", torch.int32), resid_per_seq=(lengths - per_seq * GROUP).to("cuda", torch.int32), total=int(per_seq.sum()))
    if c["padded"]:                     # left padding of a batch of unequal prompts
        pad = torch.randint(0, max(1, T // 2), (B, 1), generator=torch.Generator().manual_seed(seed + 1))
        s["mask"] = (torch.arange(T)[None] >= pad).to("cuda", torch.uint8)
    return s


def _prepare_append(c, seed):
    g, dt = _generator(seed), DTYPES[c["dtype"]]
    k = torch.stack([_keys(g, c["kv_heads"], c["tokens"], dt) for _ in range(c["batch"])])
    return {"k": k, "v": _normal(g, *k.shape, dtype=dt) if c["values"] == 4 else None}


def _model(c, seed):
    s, dt = SIZES[c["size"]], torch.bfloat16
    if c["family"] == "polar":
        from polarquant_amd.modeling_common import PolarConfig
        from polarquant_amd.modeling_llama_polar import LlamaPolarForCausalLM as cls
        cfg = PolarConfig(hidden_size=s["width"], num_attention_heads=s["heads"], num_key_value_heads=s["kv_heads"], num_hidden_layers=LAYERS,
                          intermediate_size=s["ff"], vocab_size=VOCAB, eos_token_id=[VOCAB], vbits=c["values"])
    elif c["family"] == "latent":
        from polarquant_amd.modeling_dekipel import DekipelConfig, DekipelForCausalLM as cls, DekipelLayerConfig, LatentMixerConfig
        mixers = [LatentMixerConfig(s["heads"], DIM, DIM, s["q_rank"], s["kv_rank"], DIM ** -0.5, None if i % 2 == 0 else i - 1) for i in range(LAYERS)]
        cfg = DekipelConfig(VOCAB, s["width"], [DekipelLayerConfig(m, s["ff"] * 3 // 2) for m in mixers], 1e-5, 4, 4)
    else:
        from polarquant_amd.modeling_kapudra import (DeltaMixerConfig, KapudraConfig, KapudraForCausalLM as cls, KapudraLayerConfig, MemoryMixerConfig,
                                                     ParallelMixerConfig, WindowMixerConfig)
        mixers = [ParallelMixerConfig(WindowMixerConfig(s["heads"], s["kv_heads"], DIM, DIM, s["window"], DIM ** -0.5),
                                      DeltaMixerConfig(s["heads"], s["heads"], DIM, DIM, 4, s["rank"], s["rank"]), 0.7, 0.7),
                  MemoryMixerConfig(s["memory_heads"], DIM, 2 * DIM, 15.0)]
        cfg = KapudraConfig(VOCAB, s["width"], [KapudraLayerConfig(mixers[i % 2], s["ff"]) for i in range(LAYERS)], 1e-5, math.sqrt(s["width"]), 1.0, 30.0)
    before = torch.get_default_dtype()
    torch.set_default_dtype(dt)
    try:
        with torch.device("cuda"):
            model = cls(cfg).eval()
    finally:
        torch.set_default_dtype(before)
    g = _generator(seed)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if "embed" in name:         # (scaled on reading where the family does)
                p.normal_(0.0, 1.0 / math.sqrt(s["width"]) if c["family"] == "recurrent" else 1.0, generator=g)
            elif p.dim() == 2 and p.shape[1] > 16:
                p.normal_(0.0, 1.0 / math.sqrt(p.shape[1]), generator=g)
            elif p.dim() == 2:          # filters
                p.normal_(0.0, 0.4, generator=g)
            elif "norm" in name:
                p.normal_(1.0, 0.1, generator=g)
            elif name.endswith("f_b"):  # forget gates, mostly open
                p.normal_(3.0, 1.0, generator=g)
            elif name.endswith(("A_log", "dt_bias")):           # slow and fast decays
                p.normal_(-1.0, 1.0, generator=g)
            else:
                p.normal_(0.0, 0.5, generator=g)
    return model


def prepare(case, seed):
    c = dict(case)
    if c["op"] in ("scores", "attend"):
        return dict(_prepare_cache(c, seed), case=c)
    if c["op"] == "append":
        return dict(_prepare_append(c, seed), case=c)
    g = _generator(seed + 1)
    state = {"case": c, "model": _model(c, seed), "ids": torch.randint(0, VOCAB, (c["batch"], c["tokens"]), generator=g, device="cuda"),
             "next": torch.randint(0, VOCAB, (c["batch"], 1), generator=g, device="cuda")}
    if c["op"] == "decode":             # the prompt is in the cache and the step is captured
        state["decoder"] = state["model"].graph_decoder(c["tokens"] + STEPS)
        state["decoder"].prefill(state["ids"])
        state["decoder"].step(state["next"])
    return state


# ----------------------------------------------------------------------------- one pass
def run(state):
    c = state["case"]
    if c["op"] == "scores":
        from polarquant_amd.kernel4group import attention_decode_forward_triton_impl
        return attention_decode_forward_triton_impl(state["q"], *state["cache"], rbits=c["rbits"], tbits=c["tbits"])
    if c["op"] == "attend":
        from polarquant_amd.attention import polar_decode_attention, polar_decode_attention_v4
        more = dict(attention_mask=state["mask"], rbits=c["rbits"], tbits=c["tbits"])
        if c["values"] == 4:
            return polar_decode_attention_v4(state["q"], *state["cache"], state["window"], state["v"], *state["v4"], state["groups"], state["resid"],
                                             **more)
        return polar_decode_attention(state["q"], *state["cache"], state["window"], state["v"], state["groups"], state["resid"],
                                      n_groups_per_seq=state["per_seq"], n_resid_per_seq=state["resid_per_seq"], total_groups=state["total"], **more)
    if c["op"] == "append":
        from polarquant_amd.quantize import quantize_and_pack_nbit
        from polarquant_amd.values import quantize_values
        out = quantize_and_pack_nbit(state["k"], c["rbits"], c["tbits"], eager_gpu=c["eager_gpu"])
        return (*out, *quantize_values(state["v"])) if c["values"] == 4 else out
    if c["op"] == "prompt":
        model = state["model"]
        with torch.no_grad():
            first = model(input_ids=state["ids"], num_logits_to_keep=1)
            after = model(input_ids=state["next"], past_key_values=first.past_key_values, num_logits_to_keep=1)
        return {"prompt": first.logits, "next": after.logits, "state": _float_state(c, after.past_key_values)}
    decoder = state["decoder"]
    if decoder.kv_len + 1 > decoder.max_len:            # these sequences are over: the next ones begin
        decoder.prefill(state["ids"])
    return decoder.step(state["next"])


def _float_state(c, past):
    """What the cache holds as numbers; a key code is not among them, since a key on a bin's edge may fall to either side."""
    if c["family"] == "polar":
        return [past[i][6] for i in range(LAYERS)]      # the values: all of them, or the window's where the others have 4 bits
    return [[t for t in layer[:-1] if t is not None] for layer in past]


# ----------------------------------------------------------------------------- the same in 64 bits
F64 = torch.float64


def _dequantize(c, cache, b):
    codes, rscale, rmn, tscale, tmn = [t[b] for t in cache]
    theta, rho = (codes & (2 ** c["tbits"] - 1)).to(F64), (codes >> c["tbits"]).to(F64)
    phi, r = tscale.to(F64) * (theta + 0.5) + tmn.to(F64), rscale.to(F64) * (rho + 0.5) + rmn.to(F64)
    return torch.cat([r * phi.cos(), r * phi.sin()], -1).flatten(1, 2)


def _exact_scores(c, s):
    per, out = c["heads"] // c["kv_heads"], []
    for b in range(c["batch"]):
        out.append((s["q"][b].to(F64).view(c["kv_heads"], per, DIM) @ _dequantize(c, s["cache"], b).transpose(1, 2)).flatten(0, 1)[:, None])
    return torch.stack(out)


def _exact_attend(c, s):
    per, out = c["heads"] // c["kv_heads"], []
    for b in range(c["batch"]):
        groups = s["groups"] if s["per_seq"] is None else int(s["per_seq"][b])
        resid = s["resid"] if s["per_seq"] is None else int(s["resid_per_seq"][b])
        n = groups * GROUP
        k, v = s["window"][b, :, :resid].to(F64), s["v"][b].to(F64)
        if groups:
            k = torch.cat([_dequantize(c, [t[:, :, :groups] for t in s["cache"]], b), k], 1)
        if c["values"] == 4:
            v = v[:, :resid]
            if groups:
                code, scale, lo = [t[b, :, :n] for t in s["v4"]]
                q = (code[..., None] >> torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)) & 15
                v = torch.cat([q.flatten(-2).to(F64) * scale.to(F64) + lo.to(F64), v], 1)
        else:
            v = v[:, :n + resid]
        z = s["q"][b].to(F64).view(c["kv_heads"], per, DIM) @ k.transpose(1, 2) / math.sqrt(DIM)
        if s["mask"] is not None:
            z = z.masked_fill(s["mask"][b, :n + resid] == 0, -math.inf)
        out.append((z.softmax(-1) @ v).flatten(0, 1)[:, None])
    return torch.stack(out)


def _exact_append(c, s):
    x = s["k"].unflatten(2, (-1, GROUP)).unflatten(-1, (2, PAIRS)).to(F64)
    phi = torch.atan2(x[..., 1, :], x[..., 0, :])
    out = [None]
    for v, bits in ((x.square().sum(-2).sqrt(), c["rbits"]), (torch.where(phi < 0, phi + 2 * math.pi, phi), c["tbits"])):
        lo = v.amin(-2, keepdim=True)
        out += [(v.amax(-2, keepdim=True) - lo) / 2 ** bits, lo]
    if c["values"] == 4:
        v = s["v"].to(F64)
        lo = v.amin(-1, keepdim=True)
        out += [None, (v.amax(-1, keepdim=True) - lo) / 15, lo]
    return tuple(out)


def _rms(x, w, eps, groups=1):
    n = x.unflatten(-1, (groups, -1))
    return (n / (n.square().mean(-1, keepdim=True) + eps).sqrt()).flatten(-2) * w


def _softmax_v(q, k, v, scale, slopes=None, window=None, sink=None):
    """Causal attention, q [Tq, H, d] the last of the tokens of k [T, G, d], v [T, G, dv] -> [Tq, H * dv]; some queries at a time."""
    (Tq, H, _), T = q.shape, k.shape[0]
    k, v = [t.transpose(0, 1).repeat_interleave(H // t.shape[1], 0) for t in (k, v)]
    out = []
    for i in range(0, Tq, 512):
        n = min(512, Tq - i)
        back = torch.arange(T - Tq + i, T - Tq + i + n, device="cuda")[:, None] - torch.arange(T, device="cuda")
        z = q[i:i + n].transpose(0, 1) @ k.transpose(1, 2) * scale
        if slopes is not None:
            z = z - slopes[:, None, None] * back.to(F64)
        z = z.masked_fill((back < 0) | (back >= (T if window is None else window)), -math.inf)
        m = z.amax(-1, keepdim=True)
        e = (z - m).exp_()
        total = e.sum(-1, keepdim=True)
        if sink is not None:
            total = total + (sink[:, None, None] - m).exp()
        out.append(((e @ v) / total).transpose(0, 1).flatten(1))
    return torch.cat(out)


def _conv(x, w):
    """Causal, channel by channel; the last tap meets the current token."""
    taps = w.shape[1]
    p = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
    return sum(p[j:j + len(x)] * w[:, j] for j in range(taps))


def _exact_polar(c, w, ids, tail):
    """Logits after the prompt and after each token of `tail`, which attend to the quantized cache; the layers' values."""
    s = SIZES[c["size"]]
    H, G, eps = s["heads"], s["kv_heads"], 1e-5
    bits = dict(rbits=4, tbits=4)
    caches = [None] * LAYERS
    logits, kept = [], []

    def tokens(t, first):
        x = w["model.embed_tokens.weight"][t]
        a = _angles(len(t), 500000.0, F64, first)[:, None]
        for i in range(LAYERS):
            l = "model.layers.%d." % i
            h = _rms(x, w[l + "input_layernorm.weight"], eps)
            q, k, v = [(h @ w[l + "self_attn.%s_proj.weight" % n].T).unflatten(1, (-1, DIM)) for n in "qkv"]
            q, k = _rotate(q, a.cos(), a.sin()), _rotate(k, a.cos(), a.sin())
            if caches[i] is None:
                caches[i] = [k, v]
                o = _softmax_v(q, k, v, DIM ** -0.5)
                n = len(t) // GROUP * GROUP
                if n:                   # from here on the keys are what their codes say
                    k16 = k[:n].transpose(0, 1).to(torch.bfloat16)
                    caches[i][0] = torch.cat([_dequantize(bits, [t_[None] for t_ in _quantize(k16, 4, 4, torch.bfloat16)], 0).transpose(0, 1), k[n:]])
                    if c["values"] == 4:
                        code, scale, lo = _quantize_values(v[:n].to(torch.bfloat16), torch.bfloat16)
                        nib = (code[..., None] >> torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)) & 15
                        caches[i][1] = torch.cat([nib.flatten(-2).to(F64) * scale.to(F64) + lo.to(F64), v[n:]])
            else:
                caches[i] = [torch.cat([old, new]) for old, new in zip(caches[i], (k, v))]
                o = _softmax_v(q, *caches[i], DIM ** -0.5)
            x = x + o @ w[l + "self_attn.o_proj.weight"].T
            h = _rms(x, w[l + "post_attention_layernorm.weight"], eps)
            gate, up, down = [w[l + "mlp.%s_proj.weight" % n] for n in ("gate", "up", "down")]
            x = x + (torch.nn.functional.silu(h @ gate.T) * (h @ up.T)) @ down.T
        logits.append(_rms(x[-1], w["model.norm.weight"], eps) @ w["lm_head.weight"].T)

    tokens(ids, 0)
    for j, t in enumerate(tail):
        tokens(t.view(1), len(ids) + j)
    for i in range(LAYERS):
        v = caches[i][1]
        kept.append((v if c["values"] == 16 else v[len(ids) // GROUP * GROUP:]).transpose(0, 1))
    return torch.stack(logits), kept


def _exact_latent(c, w, ids):
    """Logits of every token, the layers' states."""
    s = SIZES[c["size"]]
    H, eps = s["heads"], 1e-5
    x, latents, states = w["embed"][ids], {}, []
    for i in range(LAYERS):
        l, m = "l%d." % i, "l%d.mix." % i
        n = _rms(x, w[l + "norm1"], eps, 4)
        h = n + _conv(n, w[l + "canon1"])
        q = (_rms(h @ w[m + "dq"].T, w[m + "dq.norm"], eps) @ w[m + "uq"].T).unflatten(1, (H, -1))
        if i % 2 == 0:
            latents[i] = _rms(h @ w[m + "dkv"].T, w[m + "dkv.norm"], eps)
        cl = latents[i - i % 2]
        k, v = [(cl @ w[m + n_].T).unflatten(1, (H, -1)) for n_ in ("uk", "uv")]
        o = _softmax_v(q, k, v, DIM ** -0.5, sink=w[m + "sink"]) * torch.sigmoid(h @ w[m + "g"].T)
        x = x + _rms(o @ w[m + "o"].T, w[l + "norm1b"], eps, 4)
        n2 = _rms(x, w[l + "norm2"], eps, 4)
        h = n2 + _conv(n2, w[l + "canon2"])
        x = x + _rms((h @ w[l + "mlp.up"].T).clamp(min=0).square() @ w[l + "mlp.down"].T, w[l + "norm2b"], eps, 4)
        states.append(([latents[i]] if i % 2 == 0 else []) + [n[-3:], n2[-3:]])
    return _rms(x, w["final.norm"], eps, 4) @ w["head"].T, states


def _exact_delta(q, k, v, g, beta):
    """q, k, g [T, H, d], v [T, H, dv], beta [T, H] -> o [T, H, dv] and the last state [H, d, dv]."""
    S, out = q.new_zeros(q.shape[1], q.shape[2], v.shape[2]), torch.empty_like(v)
    for t in range(len(q)):
        S.mul_(g[t][..., None])
        u = torch.baddbmm(v[t][:, None], k[t][:, None], S, alpha=-1.0) * beta[t][:, None, None]
        S.baddbmm_(k[t][..., None], u)
        out[t] = torch.bmm(q[t][:, None], S)[:, 0]
    return out, S


def _exact_memory(q, k, v, log_i, log_f):
    """q, k [T, H, d], v [T, H, dv + 1] with a last channel of ones, gates [T, H] -> read-outs, running maxima [T, H], the last state."""
    cum = log_f.cumsum(0)
    m = cum + torch.cat([torch.zeros_like(log_i[:1]), log_i - cum]).cummax(0).values[1:]
    before = torch.cat([torch.zeros_like(m[:1]), m[:-1]])
    a, b = (log_f + before - m).exp(), (log_i - m).exp()
    S, out = q.new_zeros(q.shape[1], q.shape[2], v.shape[2]), torch.empty_like(v)
    k = k * b[..., None]
    for t in range(len(q)):
        S.mul_(a[t][:, None, None]).baddbmm_(k[t][..., None], v[t][:, None])
        out[t] = torch.bmm(q[t][:, None], S)[:, 0]
    return out, m, S


def _exact_recurrent(c, w, ids):
    """Logits of every token, the layers' states; those of a window are left out (None), being rows of a ring."""
    s = SIZES[c["size"]]
    H, G, MH, eps, T = s["heads"], s["kv_heads"], s["memory_heads"], 1e-5, len(ids)
    silu, softplus = torch.nn.functional.silu, torch.nn.functional.softplus
    x, states = w["embed"][ids] * math.sqrt(s["width"]), []
    for i in range(LAYERS):
        l = "l%d." % i
        h = _rms(x, w[l + "norm1"], eps)
        if i % 2 == 0:
            p = l + "mix.left."
            q, k = [_rms(h @ w[p + n].T, w[p + n + ".norm"], eps).unflatten(1, (-1, DIM)) for n in "qk"]
            slopes = torch.tensor([2.0 ** (-8.0 * (j + 1) / H) for j in range(H)], dtype=F64, device="cuda")
            y = 0.7 * _softmax_v(q, k, (h @ w[p + "v"].T).unflatten(1, (-1, DIM)), DIM ** -0.5, slopes, s["window"]) @ w[p + "o"].T
            p = l + "mix.right."
            lin = [h @ w[p + n].T for n in "qkv"]
            q, k, v = [silu(_conv(t, w[p + n + ".conv"])).unflatten(1, (-1, DIM)) for n, t in zip("qkv", lin)]
            q, k = [t / (t.square().sum(-1, keepdim=True) + 1e-6).sqrt() for t in (q, k)]
            a = softplus(h @ w[p + "a1"].T @ w[p + "a2"].T + w[p + "dt_bias"]).unflatten(1, (H, DIM))
            o, S = _exact_delta(q * DIM ** -0.5, k, v, (-w[p + "A_log"].exp()[:, None] * a).exp(), torch.sigmoid(h @ w[p + "b"].T))
            y = y + 0.7 * (_rms(o, w[p + "norm"], eps).flatten(1) * torch.sigmoid(h @ w[p + "g1"].T @ w[p + "g2"].T)) @ w[p + "o"].T
            states.append([None, None, torch.cat(lin, 1)[-3:], S.transpose(1, 2)])
        else:
            p = l + "mix."
            q, k, v = [(h @ w[p + n].T).unflatten(1, (MH, -1)) for n in "qkv"]
            cap = lambda z: 15.0 * torch.tanh(z / 15.0)
            log_i, log_f = cap(h @ w[p + "i"].T + w[p + "i.b"]), -softplus(-cap(h @ w[p + "f"].T + w[p + "f.b"]))
            o, m, S = _exact_memory(q * DIM ** -0.5, k, torch.cat([v, torch.ones_like(v[..., :1])], -1), log_i, log_f)
            o = o[..., :-1] / (torch.maximum(o[..., -1].abs(), (-m).exp())[..., None] + 1e-6)
            y = (_rms(o, 1.0, eps).flatten(1) * w[p + "norm"] * torch.sigmoid(h @ w[p + "g"].T)) @ w[p + "o"].T
            states.append([S.transpose(1, 2), m[-1][:, None].expand(MH, (2 * DIM + 16) // 16)])
        gate, up, down = [w[l + "mlp." + n] for n in ("gate", "up", "down")]
        x = x + y + (torch.nn.functional.gelu(h @ gate.T, approximate="tanh") * (h @ up.T)) @ down.T
    z = _rms(x, w["final.norm"], eps) @ w["head"].T
    return 30.0 * torch.tanh(z / 30.0), states


def _exact_model(c, s):
    """A prompt's logits, those of the token after it (decode: of the second one), and the cache as `run` returns it."""
    named = dict(s["model"].named_parameters()) if c["family"] == "polar" else s["model"].checkpoint_tensors()
    w = {n: p.detach().to(F64) for n, p in named.items()}
    s.pop("decoder", None)
    tail = 2 if c["op"] == "decode" else 1
    rows = []
    for b in range(c["batch"]):
        if c["family"] == "polar":
            logits, state = _exact_polar(c, w, s["ids"][b], [s["next"][b]] * tail)
            rows.append((logits[0], logits[-1], state))
        else:
            ids = torch.cat([s["ids"][b]] + [s["next"][b]] * tail)
            z, state = (_exact_latent if c["family"] == "latent" else _exact_recurrent)(c, w, ids)
            rows.append((z[c["tokens"] - 1], z[-1], state))

    def join(parts):
        if isinstance(parts[0], list):
            return [join(list(p)) for p in zip(*parts)]
        return None if parts[0] is None else torch.stack(parts)

    first, after, state = [join(list(p)) for p in zip(*rows)]
    return after[:, None] if c["op"] == "decode" else {"prompt": first[:, None], "next": after[:, None], "state": state}


@torch.no_grad()
def exact(case, seed):
    c = dict(case)
    s = prepare(dict(c, op="prompt") if c["op"] == "decode" else c, seed)
    return {"scores": _exact_scores, "attend": _exact_attend, "append": _exact_append}.get(c["op"], _exact_model)(c, s)


# ----------------------------------------------------------------------------- accounts
def _weights(c):
    """Elements of the layers' matrices and of the head."""
    s = SIZES[c["size"]]
    W, H, G, F = s["width"], s["heads"] * DIM, s["kv_heads"] * DIM, s["ff"]
    if c["family"] == "polar":
        n = LAYERS * (W * (2 * H + 2 * G) + 3 * W * F)
    elif c["family"] == "latent":
        n = LAYERS * (W * (s["q_rank"] + 2 * H) + s["q_rank"] * H + 2 * s["kv_rank"] * H + 3 * W * F) + (LAYERS + 1) // 2 * W * s["kv_rank"]
    else:
        parallel = W * (2 * H + 2 * G) + W * 4 * H + W * (2 * s["rank"] + s["heads"]) + 2 * s["rank"] * H
        n = parallel + W * s["memory_heads"] * DIM * (2 + 3 * 2) + LAYERS * 3 * W * F
    return n, W * VOCAB


def work(case):
    c = dict(case)
    B, T = c["batch"], c["tokens"]
    if c["op"] in ("scores", "attend"):
        N, Nk = c["heads"], c["kv_heads"]
        per_key = PAIRS + 4 * PAIRS * 2 / GROUP
        if c["op"] == "scores":
            return {"bytes": B * (Nk * T * per_key + N * T * 4 + N * DIM * 2), "flops": 2 * B * N * T * DIM}
        tokens = B * T * (17 / 32 if c["ragged"] else 1)
        groups = (T - 1) // GROUP * GROUP * tokens / T
        value = DIM * 2 if c["values"] == 16 else DIM // 2 + 4
        return {"bytes": Nk * (groups * (per_key + value) + (tokens - groups) * DIM * 4) + B * N * DIM * 4, "flops": 4 * N * tokens * DIM}
    if c["op"] == "append":
        per = DIM * 2 + PAIRS + 4 * PAIRS * 2 / GROUP + (DIM * 2 + DIM // 2 + 4 if c["values"] == 4 else 0)
        return {"bytes": B * c["kv_heads"] * T * per, "flops": 0}
    s = SIZES[c["size"]]
    n, head = _weights(c)
    H = s["heads"]
    if c["op"] == "prompt":
        keys = T * T / 2                # pairs of query and key
        if c["family"] == "recurrent":
            seen = min(T, s["window"])
            keys = (seen * (T - seen) + seen * seen / 2) / LAYERS
        return {"bytes": 2 * (n + head) + 4 * B * T * s["width"], "flops": 2 * B * T * n + 4 * LAYERS * B * keys * H * DIM + 2 * B * head}
    if c["family"] == "polar":
        cache = LAYERS * B * T * s["kv_heads"] * (PAIRS + 4 + (DIM * 2 if c["values"] == 16 else DIM // 2 + 4))
    elif c["family"] == "latent":
        cache = LAYERS * B * T * s["kv_rank"] * 2
    else:                               # windows are read; states are read and written
        cache = B * (min(T, s["window"]) * s["kv_heads"] * DIM * 4 + (H * DIM * DIM + s["memory_heads"] * DIM * (2 * DIM + 1)) * 8)
    return {"bytes": 2 * (n + head) + cache, "flops": 2 * B * (n + head)}


def tolerance(case):
    """Scores are float32 sums of float32 products.  Attention rounds the softmax weights and its result to 16 bits.  Codes and
    their constants are defined bit for bit.  Models round every activation to bfloat16."""
    if case["op"] == "append":
        return "exact"
    if case["op"] == "scores":
        return {"rel": 1e-5, "max": 1e-4}
    if case["op"] == "attend":
        return {"rel": 2e-3, "max": 2e-2} if case["dtype"] == "float16" else {"rel": 1e-2, "max": 8e-2}
    return {"rel": 2.5e-2, "max": 0.8}
