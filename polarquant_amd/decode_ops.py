"""Fused elementwise steps of one decode layer (HIP): RoPE + cache append, residual add + RMS norm,
SiLU * up.  Each replaces a chain of 8-12 eager launches on a [B, 1, hidden] activation
(reference: models/modeling_llama_polar.py:47-59,77,98 and the decoder layer :456-486)."""
from __future__ import annotations

from typing import Optional

import torch

from . import _ffi
from .kernel4group import _dtype_code, _on_device, _stream_ptr


def _gpu(t: torch.Tensor):
    if not t.is_cuda:
        raise RuntimeError("polarquant_amd: the fused decode ops need tensors on the GPU (no CPU fallback)")


def rope_append(q_lin: torch.Tensor, k_lin: torch.Tensor, v_lin: torch.Tensor, cos_table: torch.Tensor,
                sin_table: torch.Tensor, pos: torch.Tensor, k_dst: torch.Tensor, k_row: torch.Tensor,
                v_dst: torch.Tensor, v_row: torch.Tensor, n_heads: int, n_kv_heads: int) -> torch.Tensor:
    """q_lin [B,1,N*128], k_lin / v_lin [B,1,Nk*128] (projection outputs of the new token; each may be a
    slice along the last dim of one fused projection output: unit element stride, any batch stride);
    cos/sin tables [rows,128]; pos, k_row, v_row: int64 tensors of one element on the device.
    Writes the rotated key into k_dst[:, :, k_row] and the value into v_dst[:, :, v_row]
    ([B,Nk,rows,128] each); returns the rotated query [B,N,1,128]."""
    _gpu(q_lin)
    B = q_lin.shape[0]
    assert q_lin.stride(-1) == 1 and k_lin.stride(-1) == 1 and v_lin.stride(-1) == 1
    assert k_lin.stride(0) == v_lin.stride(0) or B == 1
    assert k_dst.is_contiguous() and v_dst.is_contiguous() and cos_table.is_contiguous() and sin_table.is_contiguous()
    assert pos.dtype == k_row.dtype == v_row.dtype == torch.int64
    assert q_lin.shape[-1] == n_heads * 128 and k_lin.shape[-1] == n_kv_heads * 128 == v_lin.shape[-1] and q_lin.numel() == B * n_heads * 128
    assert k_dst.shape[:2] == (B, n_kv_heads) == v_dst.shape[:2] and k_dst.shape[3] == 128 == v_dst.shape[3]
    q_out = torch.empty((B, n_heads, 1, 128), dtype=q_lin.dtype, device=q_lin.device)
    with _on_device(q_lin.device):
        rc = _ffi.lib().call.pq_rope_append(q_lin, k_lin, v_lin, cos_table, sin_table, cos_table.shape[0], pos, q_out, k_dst, k_dst.shape[2], k_row,
                                            v_dst, v_dst.shape[2], v_row, B, n_heads, n_kv_heads, _dtype_code(q_lin),
                                            q_lin.stride(0), k_lin.stride(0), _stream_ptr(q_lin.device))
    _ffi.check(rc, "pq_rope_append")
    return q_out


STEP_NORM_ROWS, STEP_NORM_MAX = 1023, 8192      # rows and elements of them that `embed_rmsnorm` and a norm with counters take


def embed_rmsnorm(table: torch.Tensor, ids: torch.Tensor, weight: torch.Tensor, eps: float):
    """(table[ids], weight * rms_norm of it); ids int64, outside of the table they count as its nearest row."""
    _gpu(table)
    hidden = table.shape[1]
    assert table.is_contiguous() and weight.is_contiguous() and weight.dtype == table.dtype and weight.numel() == hidden
    assert ids.is_contiguous() and ids.dtype == torch.int64 and ids.device == table.device
    x = torch.empty(tuple(ids.shape) + (hidden,), dtype=table.dtype, device=table.device)
    y = torch.empty_like(x)
    with _on_device(table.device):
        rc = _ffi.lib().call.pq_embed_rmsnorm(table, ids, table.shape[0], weight, y, x, ids.numel(), hidden, float(eps), _dtype_code(table),
                                              _stream_ptr(table.device))
    _ffi.check(rc, "pq_embed_rmsnorm")
    return x, y


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float, residual: Optional[torch.Tensor] = None,
            sum_out: Optional[torch.Tensor] = None, counters: Optional[torch.Tensor] = None,
            increments: Optional[torch.Tensor] = None) -> torch.Tensor:
    """weight * rms_norm(x), or of x + residual (the sum, rounded to the dtype, goes to sum_out,
    which may be x itself).  counters += increments (int32) in the same launch, for up to STEP_NORM_ROWS rows of STEP_NORM_MAX."""
    _gpu(x)
    hidden = x.shape[-1]
    assert x.is_contiguous() and weight.is_contiguous() and weight.dtype == x.dtype and weight.numel() == hidden
    if residual is not None:
        assert residual.is_contiguous() and residual.shape == x.shape and residual.dtype == x.dtype
    if sum_out is not None:
        assert sum_out.is_contiguous() and sum_out.shape == x.shape and sum_out.dtype == x.dtype
    y = torch.empty_like(x)
    if counters is not None:
        assert counters.is_contiguous() and increments.is_contiguous() and counters.dtype == increments.dtype == torch.int32
        assert counters.shape == increments.shape and counters.device == increments.device == x.device
        with _on_device(x.device):
            rc = _ffi.lib().call.pq_rmsnorm_advance(x, residual, weight, y, sum_out, x.numel() // hidden, hidden, float(eps), counters, increments,
                                                    counters.numel(), _dtype_code(x), _stream_ptr(x.device))
        _ffi.check(rc, "pq_rmsnorm_advance")
        return y
    with _on_device(x.device):
        rc = _ffi.lib().call.pq_rmsnorm(x, residual, weight, y, sum_out, x.numel() // hidden, hidden, float(eps), _dtype_code(x),
                                        _stream_ptr(x.device))
    _ffi.check(rc, "pq_rmsnorm")
    return y


def silu_mul(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up; gate and up [..., cols] with unit element stride and a common row stride (they
    may be the two halves of one fused projection output)."""
    _gpu(gate)
    cols = gate.shape[-1]
    assert gate.shape == up.shape and gate.dtype == up.dtype and gate.stride(-1) == 1 and up.stride(-1) == 1
    rows = gate.numel() // cols
    stride = gate.stride(-2) if gate.dim() > 1 else cols
    assert up.dim() == gate.dim() and (up.dim() == 1 or up.stride(-2) == stride)
    assert gate.dim() <= 2 or all(gate.stride(i) == gate.stride(i + 1) * gate.shape[i + 1] for i in range(gate.dim() - 2)), \
        "rows must be evenly spaced"
    y = torch.empty(gate.shape, dtype=gate.dtype, device=gate.device)
    esz = gate.element_size()
    with _on_device(gate.device):
        for r0 in range(0, rows, 65535):          # one launch covers at most 65535 rows (a prompt has more)
            n = min(65535, rows - r0)
            rc = _ffi.lib().call.pq_silu_mul(gate.data_ptr() + r0 * stride * esz, up.data_ptr() + r0 * stride * esz,
                                        y.data_ptr() + r0 * cols * esz, n, cols, stride, _dtype_code(gate),
                                        _stream_ptr(gate.device))
            _ffi.check(rc, "pq_silu_mul")
    return y


def linear_small_m(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None,
                   up_weight: Optional[torch.Tensor] = None) -> torch.Tensor:
    """`F.linear(x, weight, bias)` for at most 16 rows (x [..., K] with up to 16 leading elements, unit
    element stride, one row stride), streamed through the weight-streaming kernel.  With `up_weight`:
    the gated MLP input `silu(x @ weight.T) * (x @ up_weight.T)` in one launch (no bias)."""
    _gpu(x)
    K = x.shape[-1]
    N = weight.shape[0]
    x2 = x.reshape(-1, K)
    M = x2.shape[0]
    assert weight.is_contiguous() and weight.shape == (N, K) and weight.dtype == x.dtype and x2.stride(1) == 1
    if up_weight is not None:
        assert up_weight.is_contiguous() and up_weight.shape == weight.shape and up_weight.dtype == x.dtype
    if bias is not None:
        assert bias.is_contiguous() and bias.numel() == N and bias.dtype == x.dtype
    y = torch.empty(x.shape[:-1] + (N,), dtype=x.dtype, device=x.device)
    with _on_device(x.device):
        rc = _ffi.lib().call.pq_linear_small_m(x2, x2.stride(0) if M > 1 else K, weight, up_weight, bias, y, N, M, N, K, _dtype_code(x),
                                               _stream_ptr(x.device))
    _ffi.check(rc, "pq_linear_small_m")
    return y


def qkv_rope_append(x: torch.Tensor, w_qkv: torch.Tensor, b_qkv: Optional[torch.Tensor], cos_table: torch.Tensor,
                    sin_table: torch.Tensor, pos: torch.Tensor, k_dst: torch.Tensor, k_row: torch.Tensor,
                    v_dst: torch.Tensor, v_row: torch.Tensor, n_heads: int, n_kv_heads: int) -> torch.Tensor:
    """`linear_small_m(x, w_qkv, b_qkv)` followed by `rope_append(...)` in one launch, bit-identical to the pair:
    x [B <= 8, 1, K]; w_qkv [(N + 2 Nk) * 128, K] (q, k, v heads in that order); returns the rotated query
    [B, N, 1, 128], writes the rotated key into k_dst[:, :, k_row] and the value into v_dst[:, :, v_row]."""
    _gpu(x)
    K = x.shape[-1]
    x2 = x.reshape(-1, K)
    B = x2.shape[0]
    assert w_qkv.is_contiguous() and w_qkv.shape == ((n_heads + 2 * n_kv_heads) * 128, K) and w_qkv.dtype == x.dtype
    assert x2.stride(1) == 1 and (b_qkv is None or (b_qkv.is_contiguous() and b_qkv.numel() == w_qkv.shape[0] and b_qkv.dtype == x.dtype))
    assert k_dst.is_contiguous() and v_dst.is_contiguous() and cos_table.is_contiguous() and sin_table.is_contiguous()
    assert pos.dtype == k_row.dtype == v_row.dtype == torch.int64
    assert k_dst.shape[:2] == (B, n_kv_heads) == v_dst.shape[:2] and k_dst.shape[3] == 128 == v_dst.shape[3]
    q_out = torch.empty((B, n_heads, 1, 128), dtype=x.dtype, device=x.device)
    with _on_device(x.device):
        rc = _ffi.lib().call.pq_qkv_rope_append(x2, x2.stride(0) if B > 1 else K, w_qkv, b_qkv, B, K, _dtype_code(x), cos_table, sin_table,
                                                cos_table.shape[0], pos, q_out, k_dst, k_dst.shape[2], k_row, v_dst, v_dst.shape[2], v_row,
                                                n_heads, n_kv_heads, _stream_ptr(x.device))
    _ffi.check(rc, "pq_qkv_rope_append")
    return q_out


def normed_depth(K: int, behind: bool) -> bool:
    """Depths that the products before (`linear_residual`) and behind (`gated_normed`, `qkv_rope_append_normed`) a shared norm take."""
    return K >= 256 and K % (512 if K >= 8192 else 256) == 0 and (not behind or K <= 4096 or K == 8192)


def linear_residual(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], stream: torch.Tensor, norm_weight: torch.Tensor):
    """`stream += linear_small_m(x, weight, bias)` in place and the first half of the norm of it that follows: `stream * norm_weight` and the
    sums of squares of every 16 columns, for `gated_normed` or `qkv_rope_append_normed`.  bfloat16, up to 8 rows, `normed_depth(K, False)`."""
    _gpu(x)
    N, K = weight.shape
    x2 = x.reshape(-1, K)
    M = x2.shape[0]
    assert weight.is_contiguous() and weight.dtype == x.dtype and x2.stride(1) == 1
    assert bias is None or (bias.is_contiguous() and bias.numel() == N and bias.dtype == x.dtype)
    assert stream.is_contiguous() and stream.numel() == M * N and stream.dtype == x.dtype
    assert norm_weight.is_contiguous() and norm_weight.numel() == N and norm_weight.dtype == x.dtype
    xw = torch.empty_like(stream)
    part = torch.empty((M, N // 16), dtype=torch.float32, device=x.device)
    with _on_device(x.device):
        rc = _ffi.lib().call.pq_linear_residual(x2, x2.stride(0) if M > 1 else K, weight, bias, M, N, K, _dtype_code(x), stream, norm_weight, xw, part,
                                                _stream_ptr(x.device))
    _ffi.check(rc, "pq_linear_residual")
    return xw, part


def gated_normed(half, eps: float, weight: torch.Tensor, up_weight: torch.Tensor) -> torch.Tensor:
    """`linear_small_m(norm, weight, up_weight=up_weight)` of the norm whose first half `linear_residual` returned: the row's factor is applied
    to the sums instead of to each element, one rounding less.  `normed_depth(K, True)`."""
    xw, part = half
    N, K = weight.shape
    M = part.shape[0]
    assert weight.is_contiguous() and up_weight.is_contiguous() and up_weight.shape == weight.shape and weight.dtype == up_weight.dtype == xw.dtype
    assert xw.is_contiguous() and xw.numel() == M * K and part.is_contiguous() and part.shape[1] * 16 == K and part.dtype == torch.float32
    y = torch.empty(xw.shape[:-1] + (N,), dtype=xw.dtype, device=xw.device)
    with _on_device(xw.device):
        rc = _ffi.lib().call.pq_gated_normed(xw, part, eps, weight, up_weight, y, M, N, K, _dtype_code(xw), _stream_ptr(xw.device))
    _ffi.check(rc, "pq_gated_normed")
    return y


def qkv_rope_append_normed(half, eps: float, w_qkv: torch.Tensor, b_qkv: Optional[torch.Tensor], cos_table: torch.Tensor,
                           sin_table: torch.Tensor, pos: torch.Tensor, k_dst: torch.Tensor, k_row: torch.Tensor,
                           v_dst: torch.Tensor, v_row: torch.Tensor, n_heads: int, n_kv_heads: int) -> torch.Tensor:
    """`qkv_rope_append` of the norm whose first half `linear_residual` returned, as `gated_normed`."""
    xw, part = half
    B, K = part.shape[0], w_qkv.shape[1]
    assert w_qkv.is_contiguous() and w_qkv.shape == ((n_heads + 2 * n_kv_heads) * 128, K) and w_qkv.dtype == xw.dtype
    assert xw.is_contiguous() and xw.numel() == B * K and part.is_contiguous() and part.shape[1] * 16 == K and part.dtype == torch.float32
    assert b_qkv is None or (b_qkv.is_contiguous() and b_qkv.numel() == w_qkv.shape[0] and b_qkv.dtype == xw.dtype)
    assert k_dst.is_contiguous() and v_dst.is_contiguous() and cos_table.is_contiguous() and sin_table.is_contiguous()
    assert pos.dtype == k_row.dtype == v_row.dtype == torch.int64
    assert k_dst.shape[:2] == (B, n_kv_heads) == v_dst.shape[:2] and k_dst.shape[3] == 128 == v_dst.shape[3]
    q_out = torch.empty((B, n_heads, 1, 128), dtype=xw.dtype, device=xw.device)
    with _on_device(xw.device):
        rc = _ffi.lib().call.pq_qkv_rope_append_normed(xw, part, eps, w_qkv, b_qkv, B, K, _dtype_code(xw), cos_table, sin_table, cos_table.shape[0], pos,
                                                       q_out, k_dst, k_dst.shape[2], k_row, v_dst, v_dst.shape[2], v_row, n_heads, n_kv_heads,
                                                       _stream_ptr(xw.device))
    _ffi.check(rc, "pq_qkv_rope_append_normed")
    return q_out


def rope_qk(q_lin: torch.Tensor, k_lin: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, n_heads: int, n_kv_heads: int):
    """`apply_rotary_pos_emb` on projection outputs in one launch, bit-identical to the eager ops: q_lin [B,L,N*128],
    k_lin [B,L,Nk*128] (unit element stride, uniform token stride), cos / sin [1 or B, L, 128] in the same dtype.
    Returns (q [B,N,L,128], k [B,Nk,L,128]) as transposed views of [B,L,heads,128] tensors, the layout the eager
    `.view(B, L, heads, 128).transpose(1, 2)` followed by the rotation produces."""
    _gpu(q_lin)
    B, L = q_lin.shape[0], q_lin.shape[1]
    assert q_lin.shape[-1] == n_heads * 128 and k_lin.shape[-1] == n_kv_heads * 128 and k_lin.shape[:2] == (B, L)
    assert cos.shape == sin.shape and cos.shape[-2:] == (L, 128) and cos.shape[0] in (1, B) and cos.dtype == q_lin.dtype == k_lin.dtype

    def rows(t):                       # token b * L + l at (b * L + l) * token_stride, unit element stride
        def token_stride(u):
            return u.stride(1) if L > 1 else (u.stride(0) if B > 1 else u.shape[-1])
        if (t.stride(-1) != 1 or (B > 1 and L > 1 and t.stride(0) != L * t.stride(1)) or token_stride(t) % 8 != 0
                or token_stride(t) < t.shape[-1] or t.data_ptr() % 16):
            t = t.contiguous()
        return t, token_stride(t)
    q_lin, qs = rows(q_lin)
    k_lin, ks = rows(k_lin)
    cos, sin = cos.contiguous(), sin.contiguous()
    q_out = torch.empty((B, L, n_heads, 128), dtype=q_lin.dtype, device=q_lin.device)
    k_out = torch.empty((B, L, n_kv_heads, 128), dtype=q_lin.dtype, device=q_lin.device)
    with _on_device(q_lin.device):
        rc = _ffi.lib().call.pq_rope_qk(q_lin, qs, k_lin, ks, cos, sin, 0 if cos.shape[0] == 1 else L * 128, q_out, k_out, B, L, n_heads,
                                        n_kv_heads, _dtype_code(q_lin), _stream_ptr(q_lin.device))
    _ffi.check(rc, "pq_rope_qk")
    return q_out.transpose(1, 2), k_out.transpose(1, 2)
