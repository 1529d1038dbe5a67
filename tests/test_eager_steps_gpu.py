"""The eager modules' norm and gated activation: one launch each where the tensors allow it, the chain of torch operations otherwise.

Tolerance: both round to the dtype after every operation; they differ in the order of the sum of squares and in the last bit of
rsqrt / exp, so an element is at most one unit in the last place away per rounding (two roundings)."""
import pytest
import torch

from polarquant_amd.modeling_common import MLP, PolarConfig, RMSNorm

pytestmark = pytest.mark.gpu
UNIT = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}


def close(a, b, dtype):
    a, b = a.double(), b.double()
    return bool(((a - b).abs() <= 2 * UNIT[dtype] * b.abs() + 1e-6).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 1, 8), (2, 3, 128), (1, 130, 4096), (3, 1, 2056), (1, 2, 100)])       # (100: no multiple of 8)
def test_norm(shape, dtype):
    g = torch.Generator(device="cuda").manual_seed(shape[-1])
    norm = RMSNorm(shape[-1], 1e-5).to("cuda", dtype)
    x = (3 * torch.randn(*shape, generator=g, device="cuda")).to(dtype)
    with torch.no_grad():
        norm.weight.normal_(1.0, 0.3, generator=g)
        got = norm(x)
        strided = norm(torch.cat([x, x], -1)[..., :shape[-1]])                     # rows that are not contiguous
        assert torch.isnan(norm(torch.full_like(x, float("nan")))).all()
    want = norm(x)                                                                 # (gradients wanted: the torch operations)
    assert want.requires_grad and close(got, want, dtype) and close(strided, want, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("ff,bias", [(8, False), (520, True), (100, False)])
def test_gated_activation(ff, bias, dtype):
    g = torch.Generator(device="cuda").manual_seed(ff)
    mlp = MLP(PolarConfig(hidden_size=128, intermediate_size=ff, mlp_bias=bias)).to("cuda", dtype)
    x = (2 * torch.randn(2, 17, 128, generator=g, device="cuda")).to(dtype)
    with torch.no_grad():
        got = mlp(x)
    want = mlp(x).detach() if torch.is_grad_enabled() else None
    # the products' sums run over `ff` activations, each within two roundings
    assert float((got.double() - want.double()).norm() / want.double().norm()) < 2 * UNIT[dtype]


def test_norm_beyond_the_launch():
    """2^24 rows are more than one launch takes, a weight of one element is broadcast: the torch operations run."""
    g = torch.Generator(device="cuda").manual_seed(1)
    norm = RMSNorm(8, 1e-5).to("cuda", torch.bfloat16)
    few = torch.randn(1 << 10, 8, generator=g, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        many = norm(few.repeat(1 << 14, 1))
        assert bool((many.view(1 << 14, 1 << 10, 8) == many[:1 << 10]).all()) and close(many[:1 << 10], norm(few), torch.bfloat16)
        norm.weight = torch.nn.Parameter(norm.weight[:1] * 3)
        assert close(norm(few), 3 * many[:1 << 10], torch.bfloat16)
