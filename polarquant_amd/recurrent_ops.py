"""Windowed attention and recurrent mixers as HIP launches (include/polarquant_recurrent.h).  float16, bfloat16 or float32
weights and activations; scores, recurrent state and everything that enters a recurrence are float32.

Tensors called "rows" are [B * L, columns] with unit column stride: slices of a wider tensor will do."""
from __future__ import annotations

from typing import NamedTuple, Optional

import torch

from . import _ffi
from .attention import _num_cus
from .kernel4group import _on_device, _stream_ptr
from .layer_ops import _DTYPES, ConvState, _code

WINDOW_SMALL = 16          # new tokens per sequence up to which keys go to the ring before they are read
MAX_DIM = 256              # of a recurrent head
MAX_TAPS = 16
CHUNKED_TOKENS = WINDOW_SMALL + 1     # from this many tokens per sequence on, 16-bit recurrences run in chunks on the matrix cores
WORKSPACE_BYTES = 384 << 20         # of a chunked recurrence, at most


class Step(NamedTuple):
    """B sequences' next L tokens, at positions pos .. (*pos_dev .. when given), of sequences that begin at `start`."""
    B: int
    L: int
    pos: int
    pos_dev: Optional[torch.Tensor] = None
    start: Optional[torch.Tensor] = None


def _rows(t: torch.Tensor, M: int, n: int, dtype: torch.dtype) -> None:
    assert t.is_cuda and t.dtype == dtype and t.shape == (M, n) and (n == 1 or t.stride(1) == 1), (t.shape, t.stride(), t.dtype)


def _run(lib_fn, name: str, device, *args) -> None:
    with _on_device(device):
        rc = lib_fn(*args, _stream_ptr(device))
    _ffi.check(rc, name)


# ----------------------------------------------------------------------------- windowed attention
class WindowRing:
    """The last keys and values of B sequences: [B, G, cap, D] and [B, G, cap, Dv], position j in row j % cap."""

    def __init__(self, B: int, G: int, D: int, Dv: int, window: int, dtype, device):
        self.window, self.cap = window, -(-(window + WINDOW_SMALL - 1) // 64) * 64
        self.k = torch.zeros(B, G, self.cap, D, dtype=dtype, device=device)
        self.v = torch.zeros(B, G, self.cap, Dv, dtype=dtype, device=device)


def qk_norm(q, k, v, w_q, w_k, heads: int, eps: float, ring: WindowRing, step: Step):
    """Norms of q and of k over all their columns -> (q [M, H * D], k [M, G * D] or None); with few tokens k and v go to the
    ring."""
    B, G, cap, D = ring.k.shape
    M, Dv, dt = step.B * step.L, ring.v.shape[3], _code(q)
    assert B == step.B and ring.k.is_contiguous() and ring.v.is_contiguous() and ring.k.dtype == ring.v.dtype == q.dtype
    for t, n in ((q, heads * D), (k, G * D), (v, G * Dv)):
        _rows(t, M, n, q.dtype)
        assert t.stride(0) == q.stride(0)
    assert w_q.numel() == heads * D and w_k.numel() == G * D and w_q.dtype == w_k.dtype == q.dtype and w_q.is_contiguous() and w_k.is_contiguous()
    q_out = torch.empty(M, heads * D, dtype=q.dtype, device=q.device)
    k_out = None if step.L <= WINDOW_SMALL else torch.empty(M, G * D, dtype=q.dtype, device=q.device)
    _run(_ffi.recurrent_lib().call.pq_qk_norm, "pq_qk_norm", q.device, q, k, v, q.stride(0), w_q, w_k, q_out,
         k_out, ring.k, ring.v, step.pos_dev, step.pos, B, step.L, heads, G, D, Dv, cap, float(eps), dt)
    return q_out, k_out


def window_attention(q, ring: WindowRing, slopes: Optional[torch.Tensor], scale: float, step: Step, out: torch.Tensor, out_scale: float = 1.0,
                     k_new=None, v_new=None, n_splits: Optional[int] = None) -> torch.Tensor:
    """q [M, H * D] -> out rows [M, H * Dv] = out_scale * attention over the last `ring.window` positions, scores
    scale q.k - slopes[h] * distance.  k_new, v_new: rows of this call's keys and values, which are then put into the ring;
    without them the ring holds those already."""
    B, G, cap, D = ring.k.shape
    Dv, M, dt = ring.v.shape[3], step.B * step.L, _code(q)
    H = q.shape[1] // D
    assert q.is_contiguous() and q.shape == (M, H * D) and H % G == 0 and B == step.B and q.dtype == ring.k.dtype
    _rows(out, M, H * Dv, q.dtype)
    assert slopes is None or (slopes.dtype == torch.float32 and slopes.numel() == H and slopes.is_contiguous())
    if k_new is not None:
        assert step.pos_dev is None
        _rows(k_new, M, G * D, q.dtype)
        _rows(v_new, M, G * Dv, q.dtype)
    else:
        assert step.L <= WINDOW_SMALL
    lib = _ffi.recurrent_lib().call
    if k_new is not None:
        n_splits = 1
    elif n_splits is None:
        n_splits = lib.pq_window_plan(B, step.L, H, G, ring.window, _num_cus(q.device))
    nbytes = lib.pq_window_workspace_bytes(B, step.L, H, Dv, n_splits)
    ws = torch.empty(nbytes // 4, dtype=torch.float32, device=q.device) if nbytes else None
    kr, vr = (0, 0) if k_new is None else (k_new.stride(0), v_new.stride(0))
    _run(lib.pq_window_attn, "pq_window_attn", q.device, q, ring.k, ring.v, k_new, kr, v_new, vr, slopes,
         step.start, step.pos_dev, step.pos, out, out.stride(0), B, step.L, H, G, D, Dv, cap, ring.window, float(scale),
         float(out_scale), n_splits, ws, nbytes, dt)
    if k_new is not None:
        _run(lib.pq_ring_append, "pq_ring_append", q.device, k_new, kr, v_new, vr, ring.k, ring.v, step.pos, B, step.L,
             G, D, Dv, cap, dt)
    return out


# ----------------------------------------------------------------------------- gated delta rule
def _scan_workspace(delta: bool, dtype: torch.dtype, step: Step, heads: int, dim: int, device) -> Optional[torch.Tensor]:
    if dtype == torch.float32 or step.L < CHUNKED_TOKENS or step.pos_dev is not None:
        return None
    need = lambda tokens: _ffi.recurrent_lib().call.pq_scan_workspace_bytes(int(delta), step.B, heads, dim, tokens, _DTYPES[dtype])
    return torch.empty(min(need(step.L), max(WORKSPACE_BYTES, need(1))), dtype=torch.uint8, device=device)


class DeltaInputs(NamedTuple):
    q: torch.Tensor             # [M, G * dim] after convolution and silu
    k: torch.Tensor
    v: torch.Tensor             # [M, H * vdim]
    q_inv: torch.Tensor         # [M, G] float32: 1 / length, the query's also times dim^-1/2
    k_inv: torch.Tensor
    log_g: torch.Tensor         # [M, H * dim] float32
    beta: torch.Tensor          # [M, H] float32


def delta_prep(q, k, v, b, a, w_q, w_k, w_v, A_log, dt_bias, conv: ConvState, dim: int, vdim: int, step: Step) -> DeltaInputs:
    """Rows q, k [M, G * dim], v [M, H * vdim], b [M, H] of one projection, a [M, H * dim] decay input -> what the recurrence
    takes.  conv: the convolutions' last inputs, of q, k, v side by side."""
    M, dt, dev = step.B * step.L, _code(q), q.device
    H, G = b.shape[1], q.shape[1] // dim
    for t, n in ((q, G * dim), (k, G * dim), (v, H * vdim), (b, H)):
        _rows(t, M, n, q.dtype)
        assert t.stride(0) == q.stride(0)
    _rows(a, M, H * dim, q.dtype)
    taps = conv.taps
    for w, n in ((w_q, G * dim), (w_k, G * dim), (w_v, H * vdim)):
        assert w.shape == (n, taps) and w.is_contiguous() and w.dtype == q.dtype
    assert A_log.numel() == H and dt_bias.numel() == H * dim and A_log.dtype == dt_bias.dtype == q.dtype and A_log.is_contiguous() and dt_bias.is_contiguous()
    s_in, s_out = conv.targets(step.L)
    assert s_in.shape == (step.B, taps - 1, 2 * G * dim + H * vdim)
    e = lambda n, d: torch.empty(M, n, dtype=d, device=dev)
    r = DeltaInputs(e(G * dim, q.dtype), e(G * dim, q.dtype), e(H * vdim, q.dtype), e(G, torch.float32), e(G, torch.float32),
                    e(H * dim, torch.float32), e(H, torch.float32))
    has = taps > 1
    _run(_ffi.recurrent_lib().call.pq_delta_prep, "pq_delta_prep", dev, q, k, v, b, q.stride(0), a, a.stride(0), w_q,
         w_k, w_v, A_log, dt_bias, s_in if has else None, s_out if has else None, r.q, r.k,
         r.v, r.q_inv, r.k_inv, r.log_g, r.beta, step.start, step.pos_dev, step.pos, step.B, step.L, G, H,
         dim, vdim, taps, dt)
    return r


def delta_scan(x: DeltaInputs, state: torch.Tensor, step: Step) -> torch.Tensor:
    """state [B, H, vdim, dim] float32, advanced in place -> o [M, H * vdim] float32."""
    B, H, vdim, dim = state.shape
    M, dt, G = step.B * step.L, _code(x.q), x.q_inv.shape[1]
    assert state.is_contiguous() and state.dtype == torch.float32 and B == step.B and x.q.shape == (M, G * dim) and x.v.shape == (M, H * vdim)
    assert all(t.is_contiguous() for t in x) and x.log_g.shape == (M, H * dim) and x.beta.shape == (M, H)
    o = torch.empty(M, H * vdim, dtype=torch.float32, device=state.device)
    ws = _scan_workspace(True, x.q.dtype, step, H, dim, state.device)
    _run(_ffi.recurrent_lib().call.pq_delta_scan, "pq_delta_scan", state.device, x.q, x.k, x.v, x.q_inv, x.k_inv,
         x.log_g, x.beta, state, o, step.start, step.pos_dev, step.pos, B, step.L, G, H, dim, vdim,
         ws, 0 if ws is None else ws.numel(), dt)
    return o


# ----------------------------------------------------------------------------- matrix memory
def memory_gates(i, f, b_i, b_f, cap: float):
    """Rows i, f [M, H] of one projection -> (log input gate, log forget gate), float32 [M, H]."""
    M, H = i.shape
    dt = _code(i)
    _rows(i, M, H, i.dtype)
    _rows(f, M, H, i.dtype)
    assert i.stride(0) == f.stride(0) and b_i.numel() == b_f.numel() == H and b_i.dtype == b_f.dtype == i.dtype
    li, lf = [torch.empty(M, H, dtype=torch.float32, device=i.device) for _ in range(2)]
    _run(_ffi.recurrent_lib().call.pq_memory_gates, "pq_memory_gates", i.device, i, f, i.stride(0), b_i, b_f, li, lf,
         M, H, float(cap), dt)
    return li, lf


def memory_state(B: int, heads: int, dim: int, vdim: int, device):
    """A matrix memory's state at a sequence's start: matrices with the normalizer as their last row, running maxima (a copy
    for every 16 rows, so that no workgroup of a launch reads what another writes)."""
    return (torch.zeros(B, heads, vdim + 1, dim, dtype=torch.float32, device=device),
            torch.zeros(B, heads, (vdim + 16) // 16, dtype=torch.float32, device=device))


def memory_scan(q, k, v, log_i, log_f, state: torch.Tensor, m: torch.Tensor, q_scale: float, step: Step):
    """Rows q, k [M, H * dim], v [M, H * vdim] of one projection; state [B, H, vdim + 1, dim] and m as memory_state has them, advanced in
    place -> (o [M, H * vdim], den [M, H]) float32."""
    B, H, cols, dim = state.shape
    vdim, M, dt = cols - 1, step.B * step.L, _code(q)
    for t, n in ((q, H * dim), (k, H * dim), (v, H * vdim)):
        _rows(t, M, n, q.dtype)
        assert t.stride(0) == q.stride(0)
    assert state.is_contiguous() and m.is_contiguous() and state.dtype == m.dtype == torch.float32 and m.shape == (B, H, (vdim + 16) // 16) and B == step.B
    assert log_i.shape == log_f.shape == (M, H) and log_i.is_contiguous() and log_f.is_contiguous()
    o = torch.empty(M, H * vdim, dtype=torch.float32, device=q.device)
    den = torch.empty(M, H, dtype=torch.float32, device=q.device)
    ws = _scan_workspace(False, q.dtype, step, H, dim, q.device)
    _run(_ffi.recurrent_lib().call.pq_memory_scan, "pq_memory_scan", q.device, q, k, v, q.stride(0), log_i, log_f,
         state, m, o, den, float(q_scale), step.start, step.pos_dev, step.pos, B, step.L, H, dim, vdim,
         ws, 0 if ws is None else ws.numel(), dt)
    return o, den


def head_norm_gate(o: torch.Tensor, w: torch.Tensor, gate: torch.Tensor, heads: int, eps: float, out: torch.Tensor, out_scale: float = 1.0,
                   den: Optional[torch.Tensor] = None) -> torch.Tensor:
    """o [M, H * vdim] float32 -> out rows = out_scale * rmsnorm per head of o / den, times w ([vdim] or [H * vdim]), times
    sigmoid(gate rows)."""
    M, n = o.shape
    vdim, dt = n // heads, _code(gate)
    _rows(gate, M, n, gate.dtype)
    _rows(out, M, n, gate.dtype)
    assert o.is_contiguous() and o.dtype == torch.float32 and w.numel() in (vdim, n) and w.is_contiguous() and w.dtype == gate.dtype
    assert den is None or (den.is_contiguous() and den.dtype == torch.float32 and den.shape == (M, heads))
    _run(_ffi.recurrent_lib().call.pq_head_norm_gate, "pq_head_norm_gate", o.device, o, den, w, 0 if w.numel() == vdim else vdim,
         gate, gate.stride(0), out, out.stride(0), M, heads, vdim, float(eps), float(out_scale), dt)
    return out


# ----------------------------------------------------------------------------- one token a sequence
def _one_launch(step: Step, dtype: torch.dtype, *aligned) -> bool:
    """Whether a call could be the one launch of its mixer's token: a token a sequence, 16-bit dtype, operands at 16 bytes (their rows'
    strides and the sizes are the library's to judge)."""
    return step.L == 1 and dtype in (torch.float16, torch.bfloat16) and all(t.data_ptr() % 16 == 0 for t in aligned)


# A workgroup of the one launch has a head's whole state and most of a unit's registers, so that it pays while few rounds of workgroups fill
# the chip; beyond, the separate launches, with a state cut up, stream it faster.  Heads times sequences up to which it is the faster one, and
# us of the one / the separate launches in a chain of captured calls, bfloat16:
#   delta rule, 128 x 128, rank 128  4096: 123 / 131, 8192: 255 / 251;  128 x 96, rank 64  4096: 85 / 93, 8192: 218 / 202
#   memory  8 x 8  256: 5.9 / 7.5, 512: 9.0 / 7.8;  32 x 64  512: 9.1 / 10.9, 1024: 15.6 / 14.7;  64 x 128  1024: 18.6 / 21.9, 2048: 34.8 / 34.4
#           128 x 128  2048: 46.6 / 49.0, 4096: 98.8 / 93.6;  128 x 256  2048: 81 / 93, 4096: 207 / 184;  64 x 192  4096: 72 / 79, 8192: 178 / 168
DELTA_TOKEN_HEADS = 4096


def memory_token_heads(dim: int, vdim: int) -> int:
    if vdim >= 160 or dim * vdim >= 16384:
        return 4096 if dim <= 64 else 2048
    return 1024 if vdim >= 128 else 512 if vdim >= 64 else 256


def delta_token_takes(q, k, xa, xg, wa, wg, state: torch.Tensor, taps: int, out: torch.Tensor, step: Step, norm: Optional[torch.Tensor] = None,
                      conv: Optional[ConvState] = None) -> bool:
    """norm, conv: the norm's weight and the convolutions' state where they are not known to be of one head and at 8 bytes."""
    B, H, vdim, dim = state.shape
    return (_one_launch(step, q.dtype, xa, xg, wa, wg, state, out) and B * H <= DELTA_TOKEN_HEADS and q.shape[1] == k.shape[1] == H * dim
            and (norm is None or (norm.numel() == vdim and norm.data_ptr() % 8 == 0)) and (conv is None or conv.rows.data_ptr() % 8 == 0)
            and _ffi.recurrent_lib().call.pq_validate_delta_token(B, H, dim, vdim, taps, wa.shape[1], wg.shape[1], q.stride(0), out.stride(0),
                                                                  _DTYPES[q.dtype]) == 0)


def delta_token(q, k, v, b, xa, xg, wa, wg, w_q, w_k, w_v, A_log, dt_bias, norm, conv: ConvState, state: torch.Tensor, eps: float, out: torch.Tensor,
                out_scale: float, step: Step) -> torch.Tensor:
    """`delta_prep` with a = xa wa^T, `delta_scan` and `head_norm_gate` with the gate xg wg^T, of a token a sequence: rows q, k, v, b, xa,
    xg of one projection -> out rows [B, H * vdim]."""
    B, H, vdim, dim = state.shape
    dt, taps = _code(q), conv.taps
    assert B == step.B and step.L == 1 and state.is_contiguous() and state.dtype == torch.float32
    for t, n in ((q, H * dim), (k, H * dim), (v, H * vdim), (b, H), (xa, wa.shape[1]), (xg, wg.shape[1])):
        _rows(t, B, n, q.dtype)
        assert t.stride(0) == q.stride(0)
    _rows(out, B, H * vdim, q.dtype)
    for w, rows in ((wa, H * dim), (wg, H * vdim)):
        assert w.shape[0] == rows and w.is_contiguous() and w.dtype == q.dtype
    for w, n in ((w_q, H * dim), (w_k, H * dim), (w_v, H * vdim)):
        assert w.shape == (n, taps) and w.is_contiguous() and w.dtype == q.dtype
    assert A_log.numel() == H and dt_bias.numel() == H * dim and norm.numel() == vdim
    assert all(t.dtype == q.dtype and t.is_contiguous() for t in (A_log, dt_bias, norm))
    rows, same = conv.targets(1)
    assert rows is same and rows.shape == (B, taps - 1, 2 * H * dim + H * vdim)
    _run(_ffi.recurrent_lib().call.pq_delta_token, "pq_delta_token", q.device, q, k, v, b, xa, xg, q.stride(0), wa, wg, w_q, w_k, w_v, A_log, dt_bias,
         norm, rows if taps > 1 else None, state, out, out.stride(0), step.start, step.pos_dev, step.pos, B, H, dim, vdim, taps, wa.shape[1], wg.shape[1],
         float(eps), float(out_scale), dt)
    return out


def memory_token_takes(q, k, gate, norm, state: torch.Tensor, out: torch.Tensor, step: Step) -> bool:
    B, H, cols, dim = state.shape
    return (_one_launch(step, q.dtype, q, k, gate, norm, state, out) and B * H <= memory_token_heads(dim, cols - 1)
            and _ffi.recurrent_lib().call.pq_validate_memory_token(B, H, dim, cols - 1, q.stride(0), out.stride(0), _DTYPES[q.dtype]) == 0)


def memory_token(q, k, v, gate, i, f, b_i, b_f, norm, state: torch.Tensor, m: torch.Tensor, cap: float, q_scale: float, eps: float, out: torch.Tensor,
                 out_scale: float, step: Step) -> torch.Tensor:
    """`memory_gates`, `memory_scan` and `head_norm_gate` of a token a sequence: rows of one projection -> out rows [B, H * vdim]."""
    B, H, cols, dim = state.shape
    vdim, dt = cols - 1, _code(q)
    assert B == step.B and step.L == 1 and state.is_contiguous() and m.is_contiguous() and state.dtype == m.dtype == torch.float32
    assert m.shape == (B, H, (vdim + 16) // 16)
    for t, n in ((q, H * dim), (k, H * dim), (v, H * vdim), (gate, H * vdim), (i, H), (f, H)):
        _rows(t, B, n, q.dtype)
        assert t.stride(0) == q.stride(0)
    _rows(out, B, H * vdim, q.dtype)
    assert b_i.numel() == b_f.numel() == H and norm.numel() in (vdim, H * vdim)
    assert all(t.dtype == q.dtype and t.is_contiguous() for t in (b_i, b_f, norm))
    _run(_ffi.recurrent_lib().call.pq_memory_token, "pq_memory_token", q.device, q, k, v, gate, i, f, q.stride(0), b_i, b_f, norm,
         0 if norm.numel() == vdim else vdim, state, m, out, out.stride(0), step.start, step.pos_dev, step.pos, B, H, dim, vdim, float(cap), float(q_scale),
         float(eps), float(out_scale), dt)
    return out
