"""The eager modules of the polar models under everything that follows torch's operations: forward-mode differentiation (which no_grad leaves
on), vmap, traces, autocast, dispatch modes, subclasses.  Their own launches are invisible to all of these, so that the torch operations
have to run there."""
import pytest
import torch
import torch.autograd.forward_ad as fwad
from torch.utils._python_dispatch import TorchDispatchMode

from polarquant_amd import modeling_common as mc

UNIT = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}


class Counting(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.ops = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.ops.append(str(func))
        return func(*args, **(kwargs or {}))


class Functions(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class Subclass(torch.Tensor):
    pass


@torch.no_grad()
def test_what_counts_as_plain():
    x, plain, seen = torch.ones(3, 4), mc._nobody_looks_on, []
    note = lambda t: (seen.append(plain(t)), t * 2)[1]
    assert plain(x) and plain(x, torch.nn.Parameter(x)) and not plain(x, x.as_subclass(Subclass))
    with torch.device("cpu"):
        assert plain(x)
    torch.vmap(note)(x)
    torch.func.jvp(note, (x,), (x,))
    torch.func.functionalize(note)(x)
    torch.jit.trace(note, (x,), check_trace=False)
    torch.compile(note, backend="eager")(x)
    for mode in (fwad.dual_level(), Counting(), Functions(), torch.autocast("cuda", dtype=torch.bfloat16) if torch.cuda.is_available() else Counting()):
        with mode:
            seen.append(plain(x))
    with torch.enable_grad():
        seen.append(plain(x))
    assert seen and not any(seen) and plain(x)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("make", [lambda: mc.RMSNorm(64, 1e-5), lambda: mc.MLP(mc.PolarConfig(hidden_size=64, intermediate_size=32)), lambda: mc.Linear(64, 32)])
def test_symbolic_traces_scripts_and_dynamic_sizes(make, grad):
    """Neither values nor sizes are known there, so that nothing may be asked of them; a script compiles what it can see."""
    m, x = make(), torch.randn(40, 64)
    with torch.set_grad_enabled(grad):
        want = m(x)
        assert torch.equal(torch.fx.symbolic_trace(m)(x), want)
        assert torch.equal(torch.jit.script(m)(x), want)
        rows = torch.export.Dim("rows", min=2, max=4096)
        exported = torch.export.export(m, (torch.randn(3, 64),), dynamic_shapes=({0: rows},)).module()
        assert torch.equal(exported(x), want)


def modules(dtype):
    g = torch.Generator(device="cuda").manual_seed(1)
    for m in (mc.RMSNorm(256, 1e-5), mc.MLP(mc.PolarConfig(hidden_size=256, intermediate_size=512)), mc.Linear(256, 64)):
        m = m.to("cuda", dtype)
        for p in m.parameters():
            p.data.normal_(0.0, 0.1, generator=g)
        yield m, torch.randn(2, 3, 256, generator=g, device="cuda").to(dtype), torch.randn(2, 3, 256, generator=g, device="cuda").to(dtype)


def close(a, b, dtype, units=8):
    return float((a.double() - b.double()).norm()) <= units * UNIT[dtype] * float(b.double().norm())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_transforms_of_the_modules(dtype):
    """Values are within the roundings of the chain (8 units), tangents as those of the float64 module."""
    for m, x, t in modules(dtype):
        with torch.no_grad():
            want = m(x)
            with fwad.dual_level():
                value, tangent = fwad.unpack_dual(m(fwad.make_dual(x, t)))
            assert tangent is not None and close(value, want, dtype)
            exact = torch.func.jvp(lambda z: torch.func.functional_call(m, {n: p.double() for n, p in m.named_parameters()}, (z,)), (x.double(),), (t.double(),))[1]
            if not isinstance(m, mc.RMSNorm):           # (the norm computes in float32 whatever it is given)
                assert close(tangent, exact, dtype, 16)
            if isinstance(m, mc.RMSNorm):               # (a product under vmap is a batched product in the half dtype, which references avoid)
                assert close(torch.vmap(m)(x), want, dtype)
            traced = torch.jit.trace(m, (torch.zeros_like(x),), check_trace=False)
            assert close(traced(x), want, dtype)
            other = torch.float16 if dtype == torch.bfloat16 else torch.bfloat16
            if isinstance(m, mc.Linear):
                with torch.autocast("cuda", dtype=other):
                    assert m(x).dtype == other
            with Counting() as ops:
                m(x)
            assert any("mm" in o or "rsqrt" in o for o in ops.ops)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_prompt_attention_under_a_dispatch_mode(dtype):
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = [torch.randn(2, n, 70, 128, generator=g, device="cuda").to(dtype) for n in (4, 2, 2)]
    f = lambda a, b, c: mc._prefill_attention(a, b, c, None, 2, True)
    with torch.no_grad():
        want = f(q, k, v)
        with Counting() as ops:
            assert close(f(q, k, v), want, dtype)
        assert any("attention" in o for o in ops.ops)
