"""Which embedding modules the launches that read a table themselves may take the place of.  No GPU is needed: tensors said to be on one are
fake, and nothing is launched."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from polarquant_amd import layer_ops


def on_gpu(*shape, dtype=torch.bfloat16, index=0):
    with FakeTensorMode():
        return torch.empty(*shape, dtype=dtype, device="cuda:%d" % index)


def module(width=4096, dtype=torch.bfloat16):
    return torch.nn.Embedding(40, width, dtype=dtype)


def test_a_table_on_another_device_is_left_to_the_module():
    ids, w = on_gpu(2, 5, dtype=torch.int64), on_gpu(4096)
    assert not layer_ops.embeds(module(), ids, w, 4, 4)                                 # table on the host
    assert not layer_ops.embeds(module(), ids, on_gpu(4096, index=1), 4, 4)
    assert not layer_ops.embeds(module(), ids.to(torch.int32), w, 4, 4)


def test_the_launch_refuses_tensors_of_several_devices():
    ids, w, table = on_gpu(2, 5, dtype=torch.int64), on_gpu(4096), on_gpu(40, 4096)
    with pytest.raises(RuntimeError, match="GPU"):
        layer_ops.embed_norm_conv(module().weight.data, ids, 1.0, w, 4, 1e-5)
    conv, start = on_gpu(4096, 4), on_gpu(2, dtype=torch.int32, index=1)
    for args in ((ids, on_gpu(4096, index=1)), (on_gpu(2, 5, dtype=torch.int64, index=1), w)):
        with pytest.raises(AssertionError):
            layer_ops.embed_norm_conv(table, args[0], 1.0, args[1], 4, 1e-5)
    with pytest.raises(AssertionError):
        layer_ops.embed_norm_conv(table, ids, 1.0, w, 4, 1e-5, conv, layer_ops.ConvState(2, 4, 4096, "cpu"))
    with pytest.raises(AssertionError):
        layer_ops.embed_norm_conv(table, ids, 1.0, w, 4, 1e-5, start=start)


class Logged(torch.Tensor):
    pass


def test_only_a_plain_table_of_a_module_that_nobody_follows():
    takes = lambda e: layer_ops.only_looks_up(e, torch.bfloat16)
    e = module()
    assert takes(e) and takes(torch.nn.Embedding.from_pretrained(e.weight.data))
    assert not layer_ops.only_looks_up(e, torch.float16)
    for register in (torch.nn.modules.module.register_module_forward_hook, torch.nn.modules.module.register_module_forward_pre_hook):
        handle = register(lambda *a: None)
        assert not takes(e)
        handle.remove()
        assert takes(e)
    handle = e.register_forward_hook(lambda *a: None)
    assert not takes(e)
    handle.remove()
    assert not takes(torch.nn.Embedding.from_pretrained(Logged(e.weight.data)))
    own = module()
    own.forward = lambda ids: None
    assert not takes(own) and not takes(torch.nn.Embedding(40, 4096, max_norm=1.0, dtype=torch.bfloat16))
