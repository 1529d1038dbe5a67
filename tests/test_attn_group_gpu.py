"""Decode attention of few slices (attn_group_kernel: eight wavefronts per slice) at its edges, against the float64 oracle and against
the kernels that serve larger calls, which the same inputs reach through more slots than that kernel takes."""
import pytest
import torch

from oracle import polar_oracle as po
from polarquant_amd import _ffi, attention, workloads as wl
from polarquant_amd.attention import new_workspace, plan_splits, polar_decode_attention, polar_decode_attention_v4
from polarquant_amd.quantize import convert_codes6

pytestmark = pytest.mark.gpu
FEW = 320                   # slices the kernel takes (kGroupSlices)


def inputs(B, N, Nk, groups, resid, rbits, tbits, dtype, seed, cap=128):
    g = torch.Generator().manual_seed(seed)
    L = groups * 128 + resid
    k = wl.make_keys(B, Nk, L, 5e5, g, dtype) if L else torch.zeros(B, Nk, 0, 128, dtype=dtype)
    q, v = wl.make_half((B, N, 1, 128), g, dtype), wl.make_half((B, Nk, L, 128), g, dtype)
    codes = po.quantize_and_pack_nbit(k[:, :, :groups * 128].contiguous(), rbits, tbits) if groups else None
    kres = torch.zeros(B, Nk, cap, 128, dtype=dtype)
    kres[:, :, :resid] = k[:, :, groups * 128:]
    return q, codes, kres, v


def close(got, want, dtype):
    """fp16: the parity bar.  bf16: a window key's score is rounded to the dtype before it is scaled; scores reach 100 here, where half a
    unit is 0.25, so that a weight is off by up to 0.25 / sqrt(128) = 2.2 %, beside the roundings of weight and result (2^-9 each)."""
    got, want = got.double().cpu(), want.double()
    if dtype == torch.float16:
        return bool(((got - want).abs() <= 1e-3 + 1e-2 * want.abs()).all())
    return float((got - want).norm() / want.norm()) < 2.6e-2


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,N,Nk,groups,resid,rbits,tbits,masked", [
    (1, 8, 8, 0, 1, 4, 4, False), (2, 8, 2, 0, 128, 4, 4, True), (1, 7, 1, 1, 0, 4, 4, False), (1, 28, 4, 1, 17, 3, 3, True), (2, 16, 8, 2, 128, 4, 4, False),
    (1, 15, 3, 3, 127, 5, 2, True), (1, 12, 2, 5, 16, 6, 1, False), (3, 24, 3, 4, 15, 4, 4, True), (1, 32, 8, 9, 65, 4, 3, False)])
def test_against_the_oracle_and_the_other_kernels(gpu, dtype, B, N, Nk, groups, resid, rbits, tbits, masked):
    q, codes, kres, v = inputs(B, N, Nk, groups, resid, rbits, tbits, dtype, 10 * groups + resid)
    L = groups * 128 + resid
    mask = None
    if masked:
        mask = torch.ones(B, L, dtype=torch.uint8)
        mask[0, :L // 3] = 0
        mask[-1, L - 1:] = 1
    want = po.decode_attention_exact(q, kres[:, :, :resid], *(codes or [None] * 5), v, attention_mask=mask, rbits=rbits, tbits=tbits)
    dev = lambda t: None if t is None else t.to(gpu)
    cache = [dev(t) for t in codes] if codes else [None] * 5
    run = lambda **kw: polar_decode_attention(q.to(gpu), *cache, kres.to(gpu), v.to(gpu), groups, resid, attention_mask=dev(mask), rbits=rbits, tbits=tbits, **kw)
    few, many = FEW // (B * Nk), FEW // (B * Nk) + 1
    for name, got in (("default", run()), ("one slice", run(n_splits=1)), ("two groups a slice", run(n_splits=max(1, groups // 2))), ("empty slots", run(n_splits=few)),
                      ("pairs", run(n_splits=many)), ("single wavefront", run(single_wavefront=True)),
                      ("balanced", run(n_groups_per_seq=torch.full((B,), groups, dtype=torch.int32, device=gpu),
                                       n_resid_per_seq=torch.full((B,), resid, dtype=torch.int32, device=gpu)))):
        assert close(got, want, dtype), name


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_ragged_counts_and_a_long_window(gpu, dtype):
    """Per-sequence counts from nothing quantized to the capacity, and a window of more than 128 residual keys."""
    B, N, Nk, groups, cap = 4, 8, 2, 3, 300
    q, codes, _, v = inputs(B, N, Nk, groups, 0, 4, 4, dtype, 5)
    g = torch.Generator().manual_seed(6)
    kres = wl.make_half((B, Nk, cap, 128), g, dtype)
    v = torch.cat([v, wl.make_half((B, Nk, cap, 128), g, dtype)], 2).contiguous()
    nb, nr = [0, 1, 3, 2], [300, 1, 0, 129]
    got = polar_decode_attention(q.to(gpu), *[t.to(gpu) for t in codes], kres.to(gpu), v.to(gpu), 0, 0,
                                 n_groups_per_seq=torch.tensor(nb, dtype=torch.int32, device=gpu), n_resid_per_seq=torch.tensor(nr, dtype=torch.int32, device=gpu))
    for b in range(B):
        n, r = nb[b], nr[b]
        one = [t[b:b + 1, :, :n] for t in codes] if n else [None] * 5
        want = po.decode_attention_exact(q[b:b + 1], kres[b:b + 1, :, :r], *one, v[b:b + 1, :, :n * 128 + r])
        assert close(got[b:b + 1], want, dtype), b


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("resid", [511, 512, 513, 1100])
def test_slices_cut_on_the_device_of_a_long_window(gpu, dtype, resid):
    """Either side of the longest window that one slice keeps when the device cuts the slices."""
    q, codes, kres, v = inputs(1, 8, 2, 1, resid, 4, 4, dtype, 8, cap=resid)
    got = polar_decode_attention(q.to(gpu), *[t.to(gpu) for t in codes], kres.to(gpu), v.to(gpu), 1, resid, balanced=True, n_splits=20,
                                 n_groups_per_seq=torch.tensor([1], dtype=torch.int32, device=gpu),
                                 n_resid_per_seq=torch.tensor([resid], dtype=torch.int32, device=gpu))
    assert close(got, po.decode_attention_exact(q, kres, *codes, v), dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,N,Nk,groups,resid,packed", [(1, 8, 2, 1, 128, False), (2, 28, 4, 3, 17, True), (1, 8, 8, 2, 1, False), (1, 8, 1, 5, 0, True)])
def test_four_bit_values(gpu, dtype, B, N, Nk, groups, resid, packed):
    bits = 3 if packed else 4
    q, codes, kres, v = inputs(B, N, Nk, groups, resid, bits, bits, dtype, 3 * groups)
    vq = po.quantize_values_along_last_dim(v[:, :, :groups * 128].contiguous())
    vres = torch.zeros_like(kres)
    vres[:, :, :resid] = v[:, :, groups * 128:]
    want = po.decode_attention_mixed_exact(q, kres[:, :, :resid], *codes, vres[:, :, :resid], *vq, rbits=bits, tbits=bits)
    cache = [t.to(gpu) for t in codes]
    if packed:
        cache[0] = convert_codes6(cache[0], pack=True)
    run = lambda **kw: polar_decode_attention_v4(q.to(gpu), *cache, kres.to(gpu), vres.to(gpu), *[t.to(gpu) for t in vq], groups, resid, rbits=bits, tbits=bits, **kw)
    for got in (run(), run(n_splits=1), run(n_splits=FEW // (B * Nk)), run(single_wavefront=True)):
        assert close(got, want, dtype)


def test_nan_scores_stay_visible(gpu):
    """A NaN in a query reaches the head's output and no other, a masked-out sequence gives zeros."""
    q, codes, kres, v = inputs(1, 8, 2, 2, 5, 4, 4, torch.float16, 1)
    q[0, 3, 0, 7] = float("nan")
    run = lambda qq, m=None, **kw: polar_decode_attention(qq.to(gpu), *[t.to(gpu) for t in codes], kres.to(gpu), v.to(gpu), 2, 5, attention_mask=m, **kw)
    got = run(q, n_splits=1).cpu()
    assert torch.isnan(got[0, 3]).all() and not torch.isnan(got[0, [0, 1, 2, 4, 5, 6, 7]]).any()
    assert not run(torch.zeros_like(q), torch.zeros(1, 261, dtype=torch.uint8, device=gpu)).any()


@pytest.mark.parametrize("B,N,Nk,groups,resid,tbits,more,kw", [
    (1, 8, 8, 39, 5, 4, True, {}), (1, 8, 8, 40, 5, 4, False, {}),         # 312 and 320 slices: 320 with the window's, 328
    (16, 8, 8, 8, 5, 4, False, {}), (1, 8, 8, 5, 0, 4, False, {}), (1, 8, 8, 5, 1, 4, True, {}), (1, 8, 8, 5, 1, 5, False, {}), (1, 8, 8, 1, 5, 4, False, {}),
    (1, 8, 8, 5, 5, 4, False, dict(single_wavefront=True)), (1, 8, 8, 5, 5, 4, False, dict(min_groups_per_split=2))])
def test_when_the_window_has_a_slot_of_its_own(gpu, monkeypatch, B, N, Nk, groups, resid, tbits, more, kw):
    """One more slot than planned only where the kernel of few slices runs and there are keys for it; a workspace of the planned size is
    enough in any case."""
    q, codes, kres, v = inputs(B, N, Nk, groups, resid, 3, tbits, torch.float16, groups)
    want = po.decode_attention_exact(q, kres[:, :, :resid], *codes, v, rbits=3, tbits=tbits)
    args = [q.to(gpu), *[t.to(gpu) for t in codes], kres.to(gpu), v.to(gpu), groups, resid]
    plan = plan_splits(B, Nk, groups, gpu)
    assert plan == groups
    taken = []
    pick = attention._pick_workspace
    monkeypatch.setattr(attention, "_pick_workspace", lambda ws, b, n, splits, dev: (taken.append(splits), pick(ws, b, n, splits, dev))[1])
    for ws, splits in ((None, plan + more), (new_workspace(B, N, plan, gpu), plan), (new_workspace(B, N, plan + 1, gpu), plan + more)):
        assert close(polar_decode_attention(*args, rbits=3, tbits=tbits, workspace=ws, **kw), want, torch.float16)
        assert taken.pop() == splits, (ws is None, splits)
    if tbits == 4:
        plan4 = _ffi.lib().pq_decode_attn_v4_plan(B, N, Nk, groups, attention._num_cus(gpu))
        vq = po.quantize_values_along_last_dim(v[:, :, :groups * 128].contiguous())
        vres = torch.zeros_like(kres)
        vres[:, :, :resid] = v[:, :, groups * 128:]
        want = po.decode_attention_mixed_exact(q, kres[:, :, :resid], *codes, vres[:, :, :resid], *vq, rbits=3, tbits=tbits)
        got = polar_decode_attention_v4(*args[:7], vres.to(gpu), *[t.to(gpu) for t in vq], groups, resid, rbits=3, tbits=tbits,
                                        workspace=new_workspace(B, N, plan4, gpu), **kw)
        assert close(got, want, torch.float16) and taken.pop() == plan4


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_nan_scores_stay_visible_in_several_slices(gpu, dtype):
    """A head whose scores are all NaN has no maximum in any slice; its sums are NaN and have to reach the output through the merge, in
    every kernel, and no other head's."""
    B, N, Nk, groups, resid = 1, 8, 2, 6, 5
    q, codes, kres, v = inputs(B, N, Nk, groups, resid, 4, 4, dtype, 1)
    q[0, 3, 0, 7] = float("nan")
    q, cache, kres, v = q.to(gpu), [t.to(gpu) for t in codes], kres.to(gpu), v.to(gpu)
    vq, vres = [t.to(gpu) for t in po.quantize_values_along_last_dim(v[:, :, :groups * 128].contiguous().cpu())], torch.zeros_like(kres)
    counts = dict(n_groups_per_seq=torch.full((1,), groups, dtype=torch.int32, device=gpu), n_resid_per_seq=torch.full((1,), resid, dtype=torch.int32, device=gpu))
    for name, kw in (("default", {}), ("three", dict(n_splits=3)), ("one", dict(n_splits=1)), ("few", dict(n_splits=FEW // 2)), ("pairs", dict(n_splits=FEW // 2 + 1)),
                     ("single", dict(single_wavefront=True)), ("balanced", dict(counts, balanced=True)), ("balanced pairs", dict(counts, balanced=True, n_splits=FEW // 2 + 1))):
        for bits in (16, 4):
            if bits == 16:
                got = polar_decode_attention(q, *cache, kres, v, groups, resid, **kw)
            else:
                got = polar_decode_attention_v4(q, *cache, kres, vres, *vq, groups, resid, **kw)
            assert torch.isnan(got[0, 3]).all() and not torch.isnan(got[0, [0, 1, 2, 4, 5, 6, 7]]).any(), (name, bits)


@pytest.mark.parametrize("shape", [(1, 8, 2, 128), (1, 8, 0, 128), (1, 8, 3, 1, 128)])
def test_only_one_query_token_is_taken(gpu, shape):
    """Several tokens of a contiguous tensor would be read as other heads' queries."""
    q, codes, kres, v = inputs(1, 8, 2, 2, 5, 4, 4, torch.float16, 1)
    args = [*[t.to(gpu) for t in codes], kres.to(gpu)]
    vq = [t.to(gpu) for t in po.quantize_values_along_last_dim(v[:, :, :256].contiguous())]
    bad = torch.zeros(shape, dtype=torch.float16, device=gpu)
    for call in (lambda t: polar_decode_attention(t, *args, v.to(gpu), 2, 5), lambda t: polar_decode_attention_v4(t, *args, torch.zeros_like(args[-1]), *vq, 2, 5)):
        want = call(q.to(gpu))
        assert torch.equal(call(q.to(gpu).view(1, 8, 128)), want) and torch.equal(call(q.to(gpu).view(1, 8, 1, 1, 128)), want)
        with pytest.raises(RuntimeError):
            call(bad)


@pytest.mark.parametrize("N", [8, 16, 24])
@pytest.mark.parametrize("groups,resid", [(32, 0), (33, 0), (33, 1), (40, 0), (40, 1)])
def test_four_bit_values_around_a_workgroup_a_unit(gpu, N, groups, resid):
    """256 slices of 8 KV heads and more, where one or two heads per KV head change the kernel."""
    q, codes, kres, v = inputs(1, N, 8, groups, resid, 4, 4, torch.float16, groups + N)
    vq = po.quantize_values_along_last_dim(v[:, :, :groups * 128].contiguous())
    vres = torch.zeros_like(kres)
    vres[:, :, :resid] = v[:, :, groups * 128:]
    want = po.decode_attention_mixed_exact(q, kres[:, :, :resid], *codes, vres[:, :, :resid], *vq, rbits=4, tbits=4)
    args = [q.to(gpu), *[t.to(gpu) for t in codes], kres.to(gpu), vres.to(gpu), *[t.to(gpu) for t in vq], groups, resid]
    assert close(polar_decode_attention_v4(*args), want, torch.float16)
    nan = args[0].clone()
    nan[0, 1] = float("nan")
    got = polar_decode_attention_v4(nan, *args[1:])
    assert torch.isnan(got[0, 1]).all() and not torch.isnan(got[0, 2:]).any() and not torch.isnan(got[0, 0]).any()


@pytest.mark.parametrize("N,packed", [(32, False), (40, False), (64, False), (8, True), (32, True)])
@pytest.mark.parametrize("groups,resid", [(32, 0), (33, 0), (33, 1), (40, 0), (40, 1)])
def test_half_precision_values_around_a_workgroup_a_unit(gpu, N, packed, groups, resid):
    """The same, where packed codes or more than four heads per KV head change the kernel."""
    bits = 3 if packed else 4
    q, codes, kres, v = inputs(1, N, 8, groups, resid, bits, bits, torch.bfloat16, groups + N)
    want = po.decode_attention_exact(q, kres[:, :, :resid], *codes, v, rbits=bits, tbits=bits)
    codes = [t.to(gpu) for t in codes]
    if packed:
        codes[0] = convert_codes6(codes[0], True)
    assert close(polar_decode_attention(q.to(gpu), *codes, kres.to(gpu), v.to(gpu), groups, resid, rbits=bits, tbits=bits), want, torch.bfloat16)
