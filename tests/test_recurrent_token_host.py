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
