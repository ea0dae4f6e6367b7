"""Operators of recurrent layers: gate projections in fp32, the mLSTM's matrix-memory recurrence and the one with a constant
decay per head.

``MlstmState`` holds the state of every slot of one layer; ``mlstm`` runs a ragged step through it and applies the
per-head norm and output gate.  ``DecayMemoryState`` and ``decay_memory`` are the same for constant decays, ``gated_row_norm``
is what follows there.  All of it calls libminivllm_amd.so on the current torch stream."""
from __future__ import annotations

import math
from dataclasses import dataclass
from functools import lru_cache

import torch

from minivllm_amd import _C
from minivllm_amd.engine.ragged import BLOCK_ROWS

__all__ = ["DecayMemoryState", "MlstmState", "decay_memory", "gate_linear", "gated_row_norm", "mlstm"]

DEN_FLOOR = 1e-6          # added to the normaliser max(|n . q|, exp(-m))


def _ptr(t):
    return 0 if t is None else t.data_ptr()


@dataclass
class MlstmState:
    s: torch.Tensor       # (slots, H, dim, vdim) float32
    n: torch.Tensor       # (slots, H, dim)
    m: torch.Tensor       # (slots, H)

    @classmethod
    def allocate(cls, slots: int, heads: int, dim: int, vdim: int, device) -> "MlstmState":
        new = lambda *shape: torch.zeros(slots, heads, *shape, dtype=torch.float32, device=device)
        return cls(new(dim, vdim), new(dim), new())


def gate_linear(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None, split: int, cap: float) -> torch.Tensor:
    """float32 (T, N) = act(x weight^T + bias): columns below ``split`` through cap * tanh(z / cap), the others through
    logsigmoid of that.  x (T, K) and weight (N, K) in one dtype (bf16 / fp32), bias float32 (N,)."""
    _C.require_cuda(x, weight, bias)
    rows, k = x.shape
    n = weight.shape[0]
    if weight.dtype != x.dtype or weight.shape[1] != k or not weight.is_contiguous() or (k > 1 and x.stride(1) != 1):
        raise ValueError("x (T, K) with dense rows and a contiguous weight (N, K) of one dtype expected")
    if bias is not None and (bias.dtype != torch.float32 or bias.numel() != n or not bias.is_contiguous()):
        raise ValueError(f"bias must be contiguous float32 ({n},)")
    out = torch.empty((rows, n), dtype=torch.float32, device=x.device)
    st = _C.load().mvllm_gate_linear(_ptr(out), _ptr(x), x.stride(0) if rows > 1 else k, _ptr(weight), _ptr(bias), rows, n, k,
                                     split, float(cap), _C.dtype_code(x.dtype), _C.current_stream_ptr(x.device))
    _C.check(st, "gate_linear")
    return out


def chunked_takes(proj: torch.Tensor, dim: int, vdim: int) -> bool:
    """Whether the block form is built for this layer (otherwise every row goes through the recurrence in turn)."""
    return (proj.dtype == torch.bfloat16 and dim % 8 == 0 and vdim % 8 == 0 and dim <= 256 and proj.data_ptr() % 16 == 0
            and proj.shape[1] % 8 == 0 and (proj.shape[0] == 1 or proj.stride(0) % 8 == 0))


MAX_PARTS = 16            # csrc/memory_chunk.h: kMaxParts
PASS_OVER = 0.3           # ... kPassOver
CUS = 256


def chunked_output_fits(dim: int, vdim: int, gate: int, weight: torch.Tensor) -> bool:
    """Whether the block form's own norm and gate take this layer: whole heads of up to 128 x 256, but not those up to 128 columns, of
    which half a workgroup's waves would have none."""
    return dim <= 128 and 128 < vdim <= 256 and gate % 8 == 0 and weight.data_ptr() % 16 == 0


@lru_cache(maxsize=256)
def chunked_output_parts(fresh_rows: tuple, split: bool, heads: int, vdim: int) -> int:
    """How many workgroups share the rows of a head of portions that start from nothing (``fresh_rows``; none if one of them does not).

    A workgroup passes over the blocks in front of its own part, updating the state alone, at 0.3 of a block's time: with enough of them
    a portion of n blocks takes 0.3 n blocks' time instead of n, in one launch, as long as all run at once.  us in one part and
    shared, captured, heads of 128 x 256: 8 x 16 of 1024 rows 142 / 105 (2 parts), of 256 41 / 33.5; 8 heads, one portion of 128 17.6 / 16.2,
    of 305 32 / 24.  Where the step's segments are cut (``split``), those cost two more passes, each a launch, but then go on side by
    side however long a portion is: 31 us and the more, the more blocks there are in all.  us in segments (3 more than now) and shared: 7 x 8 of
    1000 rows 83 / 64.5, 4 x 16 of 1000 91.5 / 66, 2 x 16 of 800 54 / 45, 8 of 512 35.3 / 31.3, 4 x 8 of 1500 68.6 / 73, 8 of
    1024 43.5 / 51.  (Fewer columns, less state to combine: of 128 x 136, 4 x 8 of 1500 61.8 / 72, 2 x 16 of 800 48 / 45.)"""
    groups = heads * len(fresh_rows)
    blocks = max((-(-n // BLOCK_ROWS) for n in fresh_rows), default=0)
    parts = min(MAX_PARTS, CUS // max(groups, 1), blocks)
    if parts < 2:
        return 1
    if split:
        shared = 10.5 + 8.2 * PASS_OVER / (1 - (1 - PASS_OVER) ** parts) * blocks
        segments = 29 + 0.053 * (0.5 + vdim / 512) * heads * sum(-(-n // BLOCK_ROWS) for n in fresh_rows)
        if shared >= segments:
            return 1
    return parts


def chunked_output_takes(segments: int, rows: int, heads: int, dim: int, vdim: int, gate: int, weight: torch.Tensor) -> bool:
    """Whether ``rows`` of long entries in ``segments`` go through the norm and the output gate in the block form's own pass.

    A workgroup holds all columns of a head.  It takes longer per block of rows than two workgroups of the other form (9.5 us against 8), which have twice as
    many CUs while there are few of them, and saves a launch and the sums' way through memory.  us this form / the other, captured, heads of
    128 x 256: 64 segments of 200 rows and heads 40 / 36, 128 of them 44 / 48, 8 x 16 of 1024 rows 145 / 159; 96 of 100 rows 23.7 / 25.0, 80 of
    100 and of 190 23.2 / 22.9 and 32.6 / 33.7; 8 of 64, one block, 13.1 / 13.2 (and 12.4 / 20.2 where the launches are not captured and the host
    is the bound), 8 of 72 21.7 / 19.1 (20.7 / 20.2), 8 of 150 29.9 / 25.0.  Of 64 x 256: 8 of 100 rows 17.6 / 15.5 but 16.8 / 20.4 not captured."""
    return chunked_output_fits(dim, vdim, gate, weight) and (segments * heads >= 96 or rows <= (100 if dim <= 64 else BLOCK_ROWS) * segments)


def mlstm(step, proj: torch.Tensor, gates: torch.Tensor, gate_col: int, weight: torch.Tensor, state: MlstmState,
          eps: float) -> torch.Tensor:
    """The mLSTM mixer between its projections: (T, H * vdim) = rms(recurrence) * weight * sigmoid(gate).

    proj (T, *): q (H, dim) | k (H, dim) | v (H, vdim) at its start and the output gate's H * vdim columns at ``gate_col``;
    gates float32 (T, 2 H): log input and log forget gates; weight float32 (H * vdim,)."""
    _C.require_cuda(proj, gates, weight, state.s)
    slots, heads, dim, vdim = state.s.shape
    rows = proj.shape[0]
    if proj.dim() != 2 or proj.stride(1) != 1 or gate_col < heads * (2 * dim + vdim) or proj.shape[1] < gate_col + heads * vdim:
        raise ValueError("proj must hold q, k, v and, from gate_col on, the output gate")
    if gates.dtype != torch.float32 or tuple(gates.shape) != (rows, 2 * heads) or not gates.is_contiguous():
        raise ValueError(f"gates must be contiguous float32 ({rows}, {2 * heads})")
    if weight.dtype != torch.float32 or weight.numel() != heads * vdim or not weight.is_contiguous():
        raise ValueError(f"weight must be contiguous float32 ({heads * vdim},)")
    if step.num_tokens != rows:
        raise ValueError("the step's rows and proj's differ")
    dev, code = proj.device, _C.dtype_code(proj.dtype)
    stream = _C.current_stream_ptr(dev)
    stride = proj.stride(0) if rows > 1 else proj.shape[1]
    out = torch.empty((rows, heads * vdim), dtype=proj.dtype, device=dev)
    gate = proj.data_ptr() + gate_col * proj.element_size()
    lib = _C.load()
    scale = dim ** -0.5
    blocks = step.segments is not None and chunked_takes(proj, dim, vdim)
    # rows of long entries straight to their outputs, in several parts of a head's rows or in segments
    parts = 1
    if blocks and step.short_rows is not None and chunked_output_fits(dim, vdim, gate, weight):
        parts = chunked_output_parts(step.fresh_rows, step.split, heads, vdim)
    whole = parts > 1 or blocks and step.short_rows is not None and \
        chunked_output_takes(step.segments.shape[0], rows - step.short_rows, heads, dim, vdim, gate, weight)
    plain = step.short_rows if whole else rows                # rows whose norm and gate are a pass of their own
    state_of = (_ptr(state.s), _ptr(state.n), _ptr(state.m), _ptr(step.cu_seqlens), _ptr(step.state_slots), _ptr(step.positions))
    if plain:
        num = torch.empty((plain, heads, vdim), dtype=torch.float32, device=dev)
        den = torch.empty((plain, heads), dtype=torch.float32, device=dev)
        m_next = torch.empty((step.num_entries, heads), dtype=torch.float32, device=dev)
        common = (_ptr(num), _ptr(den), _ptr(m_next), _ptr(proj), stride, _ptr(gates), *state_of)
        row_by_row = step.num_short if blocks else step.num_entries
        if row_by_row:
            _C.check(lib.mvllm_mlstm_recurrent(*common, row_by_row, heads, dim, vdim, scale, DEN_FLOOR, code, stream),
                     "mlstm_recurrent")
    if blocks:
        count = step.segments.shape[0]
        nbytes = lib.mvllm_mlstm_chunked_workspace_bytes(count, heads, dim, vdim) if step.split else 0
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev) if nbytes else None
        tail = (_ptr(step.segments), count, int(step.split), heads, dim, vdim, scale, DEN_FLOOR, code, _ptr(ws), nbytes, stream)
        if parts > 1:
            portions = step.segments if step.portions is None else step.portions
            _C.check(lib.mvllm_mlstm_chunked_output_parts(
                _ptr(out), _ptr(weight), gate, float(eps), _ptr(proj), stride, _ptr(gates), *state_of, _ptr(portions), portions.shape[0],
                parts, heads, dim, vdim, scale, DEN_FLOOR, code, stream), "mlstm_chunked_output_parts")
        elif whole:
            _C.check(lib.mvllm_mlstm_chunked_output(_ptr(out), _ptr(weight), gate, float(eps), _ptr(proj), stride, _ptr(gates),
                                                    *state_of, *tail), "mlstm_chunked_output")
        else:
            _C.check(lib.mvllm_mlstm_chunked(*common, *tail), "mlstm_chunked")
    if plain:
        _C.check(lib.mvllm_mlstm_output(
            _ptr(out), _ptr(num), _ptr(den), _ptr(weight), gate, stride, float(eps), _ptr(m_next), _ptr(state.m),
            _ptr(step.cu_seqlens), _ptr(step.row_entry), _ptr(step.state_slots), plain, heads, vdim, code, stream), "mlstm_output")
    return out


@dataclass
class DecayMemoryState:
    s: torch.Tensor            # (slots, H, dim, vdim) float32
    decay: torch.Tensor        # (H,) float32
    log_decay: torch.Tensor    # its logarithm, taken in double precision

    @classmethod
    def allocate(cls, slots: int, decay: list, dim: int, vdim: int, device) -> "DecayMemoryState":
        if any(not 0.0 <= d <= 1.0 for d in decay):
            raise ValueError("decays must lie between 0 and 1")
        f32 = lambda x: torch.tensor(x, dtype=torch.float32, device=device)
        logs = [math.log(d) if d > 1e-300 else -1e4 for d in decay]          # exp(-1e4) is zero, and 0 * -1e4 is too
        return cls(torch.zeros(slots, len(decay), dim, vdim, dtype=torch.float32, device=device), f32(decay), f32(logs))


def decay_memory(step, proj: torch.Tensor, state: DecayMemoryState, silu: bool = True) -> torch.Tensor:
    """float32 (T, H * vdim): o = S^T q with S <- decay S + k v^T along every entry of the step, from the slots' states.

    proj (T, *): q (H, dim) | k (H, dim) | v (H, vdim) at its start; ``silu``: each of them through z * sigmoid(z) first."""
    _C.require_cuda(proj, state.s)
    slots, heads, dim, vdim = state.s.shape
    rows = proj.shape[0]
    if proj.dim() != 2 or proj.stride(1) != 1 or proj.shape[1] < heads * (2 * dim + vdim):
        raise ValueError("proj must hold q, k and v")
    if step.num_tokens != rows:
        raise ValueError("the step's rows and proj's differ")
    dev, code = proj.device, _C.dtype_code(proj.dtype)
    stream = _C.current_stream_ptr(dev)
    stride = proj.stride(0) if rows > 1 else proj.shape[1]
    num = torch.empty((rows, heads * vdim), dtype=torch.float32, device=dev)
    lib = _C.load()
    blocks = step.segments is not None and chunked_takes(proj, dim, vdim)
    row_by_row = step.num_short if blocks else step.num_entries
    if row_by_row:
        _C.check(lib.mvllm_decay_memory_recurrent(
            _ptr(num), _ptr(proj), stride, _ptr(state.decay), _ptr(state.s), _ptr(step.cu_seqlens), _ptr(step.state_slots),
            _ptr(step.positions), row_by_row, heads, dim, vdim, int(silu), code, stream), "decay_memory_recurrent")
    if blocks:
        count = step.segments.shape[0]
        nbytes = lib.mvllm_decay_memory_chunked_workspace_bytes(count, heads, dim, vdim) if step.split else 0
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev) if nbytes else None
        _C.check(lib.mvllm_decay_memory_chunked(
            _ptr(num), _ptr(proj), stride, _ptr(state.log_decay), _ptr(state.s), _ptr(step.cu_seqlens), _ptr(step.state_slots),
            _ptr(step.positions), _ptr(step.segments), count, int(step.split), heads, dim, vdim, int(silu), code, _ptr(ws),
            nbytes, stream), "decay_memory_chunked")
    return num


def gated_row_norm(x: torch.Tensor, weight: torch.Tensor, gate: torch.Tensor, eps: float) -> torch.Tensor:
    """rms(x) * weight * sigmoid(gate) over whole rows: x float32 (T, W) contiguous, weight float32 (W,), gate (T, W) with
    dense rows in the result's dtype."""
    _C.require_cuda(x, weight, gate)
    rows, width = x.shape
    if x.dtype != torch.float32 or not x.is_contiguous() or weight.dtype != torch.float32 or weight.numel() != width \
            or not weight.is_contiguous() or tuple(gate.shape) != (rows, width) or gate.stride(1) != 1:
        raise ValueError("x (T, W) and weight (W,) contiguous float32, gate (T, W) with dense rows expected")
    out = torch.empty((rows, width), dtype=gate.dtype, device=x.device)
    st = _C.load().mvllm_gated_row_norm(_ptr(out), width, _ptr(x), _ptr(weight), _ptr(gate), gate.stride(0) if rows > 1 else width,
                                        float(eps), rows, width, _C.dtype_code(gate.dtype), _C.current_stream_ptr(x.device))
    _C.check(st, "gated_row_norm")
    return out
