"""The C ABI's functions as builtins (csrc/pq_calls.cpp): the same answers as through ctypes, and questions that are answered only for
tensors as they should lie."""
import ctypes
import threading
import time

import pytest
import torch

from polarquant_amd import _ffi
from polarquant_amd._ffi import calls


@pytest.mark.parametrize("args", [(1, 8, 100, 256), (16, 8, 1, 256), (0, 0, 0, 0), (-1, 8, 100, 256), ((1 << 32) + 1, 8, 100, 256), (True, 8, 2 ** 40, 256)])
def test_the_same_integers_as_through_ctypes(args):
    lib = _ffi.lib()
    assert lib.call.pq_decode_attn_plan(*args) == lib.pq_decode_attn_plan(*args)
    assert lib.call.pq_decode_attn_workspace_bytes(*args[:3]) == lib.pq_decode_attn_workspace_bytes(*args[:3])


@pytest.mark.parametrize("pointer", [None, 0, 16, 17])
def test_the_same_refusals_as_through_ctypes(pointer):
    lib = _ffi.lib()
    args = [pointer] + [None] * 6 + [1, 8, 8, 4, 4, 4, 0, 0, None]                  # (a null pointer among them: never launched)
    assert lib.call.pq_decode_scores(*args) == lib.pq_decode_scores(*args) != 0
    strides = (128, 128, 128, 2)                                                    # no unit stride
    args = [16, strides, 0, 1, 1, 1, 4, 4, 0] + [16] * 5 + [1, 0, None]
    assert lib.call.pq_quantize_groups(*args) == lib.pq_quantize_groups(args[0], ctypes.cast((ctypes.c_int64 * 4)(*strides), ctypes.c_void_p), *args[2:])


def test_wrong_arguments_raise():
    call = _ffi.lib().call
    with pytest.raises(TypeError):
        call.pq_decode_attn_plan(1, 2, 3)
    for wrong in ("8", 1.5, None):
        with pytest.raises(ctypes.ArgumentError):
            call.pq_decode_attn_plan(1, wrong, 3, 4)
    with pytest.raises(ctypes.ArgumentError):
        call.pq_decode_scores("q", *[None] * 6, 1, 8, 8, 4, 4, 4, 0, 0, None)


def test_tensors_that_are_not_plain_are_left_to_the_general_path():
    q, codes, meta = torch.zeros(1, 8, 1, 128, dtype=torch.float16), torch.zeros(1, 8, 2, 128, 64, dtype=torch.uint8), torch.zeros(1, 8, 2, 1, 64, dtype=torch.float16)
    assert calls.plain_scores(q, codes, meta, meta, meta, meta) is None             # (not on a GPU)
    assert calls.plain_cache(q, codes, meta, meta, meta, meta, None, q, None, None, None, None) is None
    assert calls.plain_rows(q, 4, 8) is None and calls.plain_rows(None, 4, 8) is None
    with torch.no_grad():
        assert calls.plain_half(q) is False and calls.plain_eager(q) is True
        assert calls.plain_eager(torch.nn.Parameter(q)) is True and calls.plain_eager(q.as_subclass(type("Sub", (torch.Tensor,), {}))) is None
        with torch.device("cpu"):
            assert calls.plain_eager(q) is None                                     # (a mode: looked at more closely)
        with torch.autograd.forward_ad.dual_level():
            assert calls.plain_eager(q) is None
        seen = []
        torch.func.vmap(lambda t: (t, seen.append(calls.plain_half(t)))[0])(q)
        assert seen == [None]
    assert calls.plain_eager(q) is None                                             # (gradients are on)


def test_empty():
    like = torch.zeros(1, dtype=torch.bfloat16)
    for code, dtype in ((0, torch.bfloat16), (1, torch.uint8), (2, torch.int32), (3, torch.float32)):
        t = calls.empty(like, code, 2, 0, 3)
        assert t.shape == (2, 0, 3) and t.dtype == dtype and t.device == like.device and t.is_contiguous()
    with pytest.raises(RuntimeError):
        calls.empty(like, 0, -1)


def test_scores_want_a_query_for_every_sequence():
    from torch._subclasses.fake_tensor import FakeTensorMode
    from polarquant_amd.kernel4group import attention_decode_forward_triton_impl as scores
    with FakeTensorMode():
        q, codes, meta = [torch.zeros(*s, dtype=d, device="cuda") for s, d in (((1, 8, 1, 128), torch.float16), ((2, 8, 2, 128, 64), torch.uint8), ((2, 8, 2, 1, 64), torch.float16))]
    with pytest.raises(ValueError, match="queries"):
        scores(q, codes, meta, meta, meta, meta)


@pytest.mark.parametrize("wrong", [1 << 20, (1, 2), [1, 2], 0.5])
def test_counts_and_positions_are_tensors(wrong):
    """A number or a tuple where a count per sequence, a position or a state belongs is refused, not read as an address."""
    call = _ffi.lib().call
    nothing = [None] * 6
    for groups, resid in ((wrong, None), (None, wrong)):
        with pytest.raises(ctypes.ArgumentError):
            call.pq_decode_attn(*nothing, 1, 1, groups, None, 0, 0, resid, None, 1, None, 0, 1.0, 1, 8, 8, 4, 4, 0, 1, 1, None, 0, None, 0, None, None)
    with pytest.raises(ctypes.ArgumentError):
        _ffi.latent_lib().call.pq_latent_decode(None, None, 1, None, None, wrong, 0, None, 1, 1, 1, 64, 1.0, 1, None, 0, 0, None)
    with pytest.raises(ctypes.ArgumentError):
        _ffi.steps_lib().call.pq_embed_rows(None, wrong, 1.0, None, 1, 8, 1, 0, None)


def test_another_prototype_is_not_bound():
    """Builtins of other headers than the checkout's would hand a library arguments that are not its own."""
    lib, name = _ffi.lib(), "pq_decode_attn_plan"
    at = ctypes.cast(getattr(lib, name), ctypes.c_void_p).value
    assert calls.bind(name, at, "iiiii")(1, 8, 100, 256) == lib.pq_decode_attn_plan(1, 8, 100, 256)
    for other in ("iiii", "iiiiii", "iiiil", "iiiif", "Iiiii", ""):
        with pytest.raises(RuntimeError, match="another version"):
            calls.bind(name, at, other)
    assert calls.bind("pq_version", at, "i") is None


def test_other_threads_run_while_memory_is_allocated():
    """An allocation that takes long (1 GiB that the deterministic mode fills) does not hold the interpreter."""
    seen, over = [], threading.Event()

    def watch():
        while not over.is_set():
            seen.append(time.perf_counter())
            time.sleep(0.001)
    before = torch.are_deterministic_algorithms_enabled()
    other = threading.Thread(target=watch)
    torch.use_deterministic_algorithms(True)
    try:
        other.start()
        first = time.perf_counter()
        t = calls.empty(torch.zeros(1), 3, 1 << 28)
        last = time.perf_counter()
    finally:
        torch.use_deterministic_algorithms(before)
        over.set()
        other.join()
    assert torch.isnan(t[::1 << 20]).all()
    spent = last - first
    assert any(first + 0.1 * spent < s < last - 0.1 * spent for s in seen), spent
