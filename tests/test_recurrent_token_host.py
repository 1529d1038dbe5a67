"""Which calls of a token a sequence are one launch (recurrent_ops: `delta_token_takes`, `memory_token_takes`).  No GPU is needed."""
import pytest
import torch

from polarquant_amd import layer_ops
from polarquant_amd import recurrent_ops as ops
from polarquant_amd.recurrent_ops import Step


def at(t, elements):
    """A copy of t that lies so many elements behind an aligned address."""
    return torch.cat([t.new_zeros(elements), t.flatten()])[elements:].view(t.shape)


def delta(B=1, H=2, dim=128, vdim=128, norm=lambda t: t, conv=lambda t: t, L=1):
    h = lambda *s: torch.zeros(*s, dtype=torch.float16)
    state = ops.ConvState(B, 4, 2 * H * dim + H * vdim, "cpu")
    state._buf[0] = conv(state._buf[0])
    return ops.delta_token_takes(h(B, H * dim), h(B, H * dim), h(B, 64), h(B, 64), h(H * dim, 64), h(H * vdim, 64), torch.zeros(B, H, vdim, dim), 4,
                                 h(B, H * vdim), Step(B, L, 0), norm(h(vdim)), state)


def test_delta_rule_asks_where_its_operands_lie():
    assert delta() and delta(norm=lambda t: at(t, 4)) and delta(conv=lambda t: at(t, 2))
    assert not delta(L=2)
    for n in (1, 2, 3):
        assert not delta(norm=lambda t: at(t, n))
    assert not delta(conv=lambda t: at(t, 1))
    assert not delta(norm=lambda t: t.repeat(2))                      # a norm a head


def memory(B, H, dim, vdim):
    p = torch.empty(B, H * max(dim, vdim), dtype=torch.float16)
    q, gate = p[:, :H * dim], p[:, :H * vdim]
    return ops.memory_token_takes(q, q, gate, torch.empty(H * vdim, dtype=torch.float16), torch.empty(B, H, vdim + 1, dim), torch.empty_like(gate), Step(B, 1, 0))


@pytest.mark.parametrize("dim,vdim,heads", [(8, 8, 256), (32, 64, 512), (40, 72, 512), (64, 128, 1024), (96, 128, 1024), (128, 128, 2048), (128, 160, 2048), (64, 192, 4096),
                                            (8, 256, 4096)])
def test_memory_takes_the_side_that_is_faster(dim, vdim, heads):
    assert memory(1, 1, dim, vdim) and memory(8, heads // 8, dim, vdim) and not memory(8, heads // 8 + 1, dim, vdim) and not memory(2 * heads, 1, dim, vdim)


@pytest.mark.parametrize("dim,vdim", [(128, 128), (128, 96), (96, 96)])
def test_delta_rule_takes_the_side_that_is_faster(dim, vdim):
    assert delta(1, 1, dim, vdim) and delta(128, 32, dim, vdim) and not delta(129, 32, dim, vdim)
