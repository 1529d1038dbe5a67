"""A norm shared by the products around it (`linear_residual`, `gated_normed`, `qkv_rope_append_normed`) against the launches it replaces
and against 64 bits: splits of the depth (four ways, eight from 8192 on), two and four row tiles, one to eight rows, the narrowest and the widest norm."""
import pytest
import torch

from polarquant_amd import _ffi
from polarquant_amd.decode_ops import (gated_normed, linear_residual, linear_small_m, normed_depth, qkv_rope_append, qkv_rope_append_normed, rmsnorm)

pytestmark = pytest.mark.gpu
EPS = 1e-5


def draw(gpu, g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16).to(gpu)


def norm64(stream, w):
    x = stream.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def half(gpu, M, width, K, bias=True, seed=0):
    g = torch.Generator().manual_seed(1000 * M + width + K + seed)
    x, w, stream, nw = draw(gpu, g, M, 1, K), draw(gpu, g, width, K, scale=K ** -0.5), draw(gpu, g, M, 1, width, scale=3.0), draw(gpu, g, width)
    b = draw(gpu, g, width) if bias else None
    a = linear_small_m(x, w, b)
    want = stream + a
    h = rmsnorm(stream, nw, EPS, residual=a)
    xw, part = linear_residual(x, w, b, stream, nw)
    return stream, want, nw, h, (xw, part), g


@pytest.mark.parametrize("M", [1, 3, 8])
@pytest.mark.parametrize("width,K", [(256, 256), (512, 8192), (4096, 1024), (8192, 256), (16384, 512), (272, 768)])
def test_product_into_the_stream(gpu, M, width, K):
    """The stream and its products with the norm's weight bit for bit what the separate launches leave; sums of sixteen squares to float32."""
    stream, want, nw, _, (xw, part), _ = half(gpu, M, width, K, bias=M != 3)
    assert torch.equal(stream, want)
    assert torch.equal(xw, stream * nw)
    exact = stream.double().square().reshape(M, width // 16, 16).sum(-1)
    assert bool(((part.double() - exact).abs() <= 6 * 2.0 ** -24 * exact).all())         # four fused steps and two additions in turn, half an ulp each


def product64(stream, nw, w, bias=0.0):
    """The product of the norm in 64 bits, and how far a result in bfloat16 may be: half an ulp (2^-9) of each x w and of the result, 1 % for what
    float32 sums and the square of that add."""
    n, w = norm64(stream, nw), w.double()
    y = n @ w.T + bias
    return y, 1.01 * 2.0 ** -9 * (n.abs() @ w.abs().T + y.abs())


def within(got, separate, exact, bound):
    assert bool(((got.double() - exact).abs() <= bound).all())
    e = lambda t: ((t.double() - exact).square().mean() / exact.square().mean()).sqrt().item()
    if got.numel() >= 60000:       # (squared errors have a kurtosis of some 20: the estimates' ratio is 1 % uncertain here, several tenths for a few hundred)
        assert e(got) <= 1.05 * e(separate), (e(got), e(separate))


@pytest.mark.parametrize("M", [1, 5, 8])
@pytest.mark.parametrize("width,ff", [(256, 64), (4096, 272), (2048, 8192), (8192, 512)])
def test_gated_product(gpu, M, width, ff):
    stream, _, nw, h, hf, g = half(gpu, M, width, 256)
    gate, up = draw(gpu, g, ff, width, scale=width ** -0.5), draw(gpu, g, ff, width, scale=width ** -0.5)
    got = gated_normed(hf, EPS, gate, up)
    (gv, gb), (uv, ub) = product64(stream, nw, gate), product64(stream, nw, up)
    sv, sb = torch.nn.functional.silu(gv), 1.1 * gb                     # (silu's slope is below 1.1)
    sb = sb + 2.0 ** -9 * (sv.abs() + sb)
    bound = sb * uv.abs() + sv.abs() * ub + sb * ub
    exact = sv * uv
    within(got, linear_small_m(h, gate, up_weight=up), exact, bound + 2.0 ** -9 * (exact.abs() + bound))


@pytest.mark.parametrize("M", [1, 8])
@pytest.mark.parametrize("width,N,Nk,bias", [(512, 4, 2, True), (4096, 8, 8, False), (8192, 2, 1, True)])
def test_projections_with_rotation(gpu, M, width, N, Nk, bias):
    stream, _, nw, h, hf, g = half(gpu, M, width, 512)
    w = draw(gpu, g, (N + 2 * Nk) * 128, width, scale=width ** -0.5)
    b = draw(gpu, g, (N + 2 * Nk) * 128) if bias else None
    ang = torch.rand(9, 64, generator=g) * 6.28
    cos, sin = (torch.cat([f, f], -1).to(torch.bfloat16).to(gpu) for f in (ang.cos(), ang.sin()))
    at = lambda i: torch.tensor([i], dtype=torch.int64, device=gpu)
    outs = []
    for fused in (True, False):
        k, v = torch.zeros(M, Nk, 5, 128, dtype=torch.bfloat16, device=gpu), torch.zeros(M, Nk, 9, 128, dtype=torch.bfloat16, device=gpu)
        rest = (w, b, cos, sin, at(7), k, at(2), v, at(7), N, Nk)
        q = qkv_rope_append_normed(hf, EPS, *rest) if fused else qkv_rope_append(h, *rest)
        assert int((k != 0).any(-1).sum()) == int((v != 0).any(-1).sum()) == M * Nk          # one row of each
        outs.append(torch.cat([q[:, :, 0], k[:, :, 2], v[:, :, 7]], 1))
    y, yb = (t.reshape(M, N + 2 * Nk, 128) for t in product64(stream, nw, w, b.double() if bias else 0.0))
    c, s = cos[7].double(), sin[7].double()
    turn = lambda t, sign: torch.cat([sign * t[:, :N + Nk, 64:], t[:, :N + Nk, :64]], -1)
    exact = torch.cat([y[:, :N + Nk] * c + turn(y, -1) * s, y[:, N + Nk:]], 1)
    # the rotation: half an ulp of each of its products and of their sum
    most = lambda t: t[:, :N + Nk] * c.abs() + turn(t, 1) * s.abs()
    bound = torch.cat([most(yb) + 2.02 * 2.0 ** -9 * most(y.abs() + yb), yb[:, N + Nk:]], 1)
    within(*outs, exact, bound)


def test_what_is_not_taken(gpu):
    """float16 (the product with the weight could overflow), more than eight rows, depths without a whole split."""
    call, P = _ffi.lib(), 4096
    ok = [P, 4096, P, None, 8, 4096, 4096, 1, P, P, P, P]
    assert call.pq_validate_linear_residual(*ok) == 0
    for i, v in ((7, 0), (4, 9), (6, 320), (6, 8448), (8, None), (11, None)):
        bad = list(ok)
        bad[i] = v
        bad[1] = max(bad[1], bad[6])
        assert call.pq_validate_linear_residual(*bad) != 0, (i, v)
    ok = [P, P, P, P, P, 8, 512, 4096, 1]
    assert call.pq_validate_gated_normed(*ok) == 0
    for i, v in ((8, 0), (5, 9), (7, 4352), (7, 5120), (1, None), (3, None), (1, 4100)):
        bad = list(ok)
        bad[i] = v
        assert call.pq_validate_gated_normed(*bad) != 0, (i, v)
    for K in range(64, 20000, 64):
        assert normed_depth(K, False) == (call.pq_validate_linear_residual(P, K, P, None, 8, 4096, K, 1, P, P, P, P) == 0)
        assert normed_depth(K, True) == (call.pq_validate_gated_normed(P, P, P, P, P, 8, 512, K, 1) == 0)


# launches that the cases above leave out: rows, width, and columns of the product behind or depth of the one before
GATED_VARIANTS = [(1, 4096, 14336), (5, 4096, 14336), (8, 4096, 14336), (8, 512, 16384), (8, 4096, 8192), (8, 8192, 8192)]
INTO_VARIANTS = [(8, 8192, 8192), (8, 8192, 8704), (8, 5120, 8704), (8, 4096, 14336), (1, 8192, 4096), (8, 8192, 4096), (2, 4096, 4096), (8, 4096, 4096)]


@pytest.mark.parametrize("M,width,ff", GATED_VARIANTS)
def test_gated_product_of_every_launch(gpu, M, width, ff):
    """(From 60000 results on with the RMS error against the separate launches.)"""
    test_gated_product(gpu, M, width, ff)


@pytest.mark.parametrize("M,width,K", INTO_VARIANTS)
def test_product_into_the_stream_of_every_launch(gpu, M, width, K):
    test_product_into_the_stream(gpu, M, width, K)


def test_projections_with_rotation_error(gpu):
    """Enough results for the RMS error, at the widest norm of a depth split four ways and of one split eight ways."""
    for width in (4096, 8192):
        test_projections_with_rotation(gpu, 8, width, 56, 4, True)


@pytest.mark.parametrize("eps", [1e-5, 1e-3])
@pytest.mark.parametrize("width", [256, 2048, 4096, 8192])
def test_factor_of_a_row(gpu, width, eps):
    """The products' factor of a row by itself.  Rows of weights that hold a single one make every product exact, so that a value is r (x w)
    rounded once: the same bits as from r in 64 bits unless that lies within float32's error (2^-22) of a tie, one in 2^13.  A row's energy
    lies in one block of 16 columns, each block in turn, so that a sum that is missed changes everything; the rows are small enough that eps
    is a good part of the mean square."""
    g = torch.Generator().manual_seed(width)
    N, Nk = 1, 4
    nw = draw(gpu, g, width) + 2.0
    cols = torch.randint(0, width, ((N + 2 * Nk) * 128,), generator=g)
    w = torch.zeros((N + 2 * Nk) * 128, width, dtype=torch.bfloat16)
    w[torch.arange(len(cols)), cols] = 1.0
    gate, up = torch.zeros(512, width, dtype=torch.bfloat16), torch.zeros(512, width, dtype=torch.bfloat16)
    gate[torch.arange(512), cols[:512]] = 1.0
    up[torch.arange(512), cols[512:1024]] = 1.0
    w, gate, up = w.to(gpu), gate.to(gpu), up.to(gpu)
    cos = torch.ones(4, 128, dtype=torch.bfloat16, device=gpu)
    at = torch.zeros(1, dtype=torch.int64, device=gpu)
    rounded = lambda t: t.to(torch.bfloat16).double()
    same, total = 0, 0
    for first in range(0, width // 16, 8):
        stream = draw(gpu, g, 8, 1, width, scale=1e-3)
        for m in range(8):
            block = first + m
            stream[m, 0, 16 * block:16 * block + 16] = draw(gpu, g, 16, scale=0.2) + 0.3
        xw, part = linear_residual(torch.zeros(8, 1, 256, dtype=torch.bfloat16, device=gpu), torch.zeros(width, 256, dtype=torch.bfloat16, device=gpu), None,
                                   stream, nw)
        r64 = torch.rsqrt(stream.double().square().mean(-1) + eps)
        n64 = xw.double()[:, 0] * r64
        k, v = torch.zeros(8, Nk, 1, 128, dtype=torch.bfloat16, device=gpu), torch.zeros(8, Nk, 1, 128, dtype=torch.bfloat16, device=gpu)
        qkv_rope_append_normed((xw, part), eps, w, None, cos, torch.zeros_like(cos), at, k, at, v, at, N, Nk)
        got = gated_normed((xw, part), eps, gate, up)[:, 0]
        gv, uv = rounded(n64[:, cols[:512]]), rounded(n64[:, cols[512:1024]])
        want = [(k.reshape(8, -1), rounded(n64[:, cols[128:640]])), (v.reshape(8, -1), rounded(n64[:, cols[640:]])),
                (got, rounded(rounded(torch.nn.functional.silu(gv)) * uv))]
        for y, e in want:
            assert bool(((y.double() - e).abs() <= 2.0 ** -6 * e.abs() + 1e-30).all())          # the other neighbour of each rounding
            same += int((y.double() == e).sum())
            total += y.numel()
    assert same >= 0.995 * total, (same, total)
