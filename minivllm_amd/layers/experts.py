"""Mixture of experts: router, plan and products as operators over libminivllm_amd.so, and the feed-forward module.

The module returns the experts' results unsummed (``ExpertOutput``): whoever adds the feed-forward to the residual reads
them with their weights (``layers.fused.stream_norm``)."""
from __future__ import annotations

import ctypes
from dataclasses import dataclass
from typing import Optional

import torch
import torch.nn as nn
from torch.nn.modules.module import _has_any_global_hook

from minivllm_amd import _C
from minivllm_amd.layers.basic import Linear, SiluAndMul
from minivllm_amd.layers.recurrent import gate_linear
from minivllm_amd.models.qwen3 import Qwen3MLP, _as_built
from minivllm_amd.utils.padding import pad_to, round_up

__all__ = ["ExpertOutput", "ExpertPlan", "SparseExperts", "moe_route", "moe_route_softmax", "moe_plan", "moe_linear", "moe_linear_tiles", "interleave_gate_up"]

FEW_PAIRS = 16             # (token, choice) pairs up to which the products run without a plan ...
# ... where rows are short and no shared expert can join the launches: without one every expert has workgroups that look for its rows, with one only those that have
# some have any, and the shared expert is part of the launches.  us of a captured pass, without / with, one row, top 2: 8 experts of 256 x 512 13.1 / 16.8, 128 of them 15.9 / 19.5,
# 8 of 512 x 512 18.3 / 19.3 (with a shared expert 23.2 / 19.5); 8 of 768 x 768 23.9 / 17.8, of 128 x 2048 20.3 / 19.5, of 256 x 1024 18.8 / 17.5, 128 of them 21.9 / 19.6, eight rows
# 28.6 / 21.0; top 6 of 64 of 768 x 2048 44 / 25, top 8 of 1280 x 4096 91 / 61; 8 of 14336 x 4096 197 / 126, eight rows 512 / 387.
SHORT_ROWS = 768
_PLAIN = (nn.Parameter, torch.Tensor)


def _ptr(t):
    return 0 if t is None else t.data_ptr()


@dataclass
class ExpertOutput:
    """y[t] = sum_k weights[t, k] parts[part_row[t, k]] + sigmoid(gate[t]) shared[t]; a choice whose id is negative counts with
    inputs[t]."""
    parts: torch.Tensor                       # (pairs, >= width)
    weights: torch.Tensor                     # float32 (T, top)
    part_row: Optional[torch.Tensor] = None   # int32 (T * top,), None: pair t * top + k
    shared: Optional[torch.Tensor] = None     # (T, width)
    gate: Optional[torch.Tensor] = None       # float32 (T,), any stride; None: 1
    ids: Optional[torch.Tensor] = None        # int32 (T, top), None: every choice is an expert
    inputs: Optional[torch.Tensor] = None     # (T, >= width)


class ExpertPlan:
    """Pairs sorted by expert (device memory only; the host never learns how many rows an expert has)."""

    def __init__(self, ids: torch.Tensor, experts: int):
        self.pairs = ids.numel()
        nbytes = int(_C.load().mvllm_moe_plan_bytes(self.pairs, experts))
        self.data = torch.empty(nbytes // 4, dtype=torch.int32, device=ids.device)
        st = _C.load().mvllm_moe_plan(_ptr(self.data), nbytes, _ptr(ids), self.pairs, experts, _C.current_stream_ptr(ids.device))
        _C.check(st, "moe_plan")

    @property
    def place(self) -> torch.Tensor:
        """Sorted place of every pair."""
        return self.data[:self.pairs]


def _span(x) -> int:
    """Numbers from the first of x (rows, K) to behind the last, rows dense."""
    return (x.shape[0] - 1) * x.stride(0) + x.shape[1]


def moe_route(logits: torch.Tensor, correction: torch.Tensor | None, experts: int, top: int, groups: int = 1, keep: int = 1):
    """(ids int32 (T, top), weights float32 (T, top)) from float32 logits (T, >= experts)."""
    _C.require_cuda(logits, correction)
    if logits.dtype != torch.float32 or logits.stride(1) != 1 or logits.shape[1] < experts:
        raise ValueError("logits must be float32 with dense rows, one column per expert")
    if correction is not None and (correction.dtype != torch.float32 or correction.numel() != experts or not correction.is_contiguous()):
        raise ValueError(f"correction must be contiguous float32 ({experts},)")
    t = logits.shape[0]
    ids = torch.empty((t, top), dtype=torch.int32, device=logits.device)
    weights = torch.empty((t, top), dtype=torch.float32, device=logits.device)
    st = _C.load().mvllm_moe_route(_ptr(ids), _ptr(weights), _ptr(logits), logits.stride(0) if t > 1 else logits.shape[1],
                                   _ptr(correction), t, experts, top, groups, keep, _C.current_stream_ptr(logits.device))
    _C.check(st, "moe_route")
    return ids, weights


def moe_route_softmax(logits: torch.Tensor, correction: torch.Tensor | None, experts: int, identity: int, top: int,
                      renormalize: bool = False):
    """(ids int32 (T, top), weights float32 (T, top)): the largest softmax(logits) + correction, weighted by the softmax.  The last
    ``identity`` of the experts + identity columns stand for no expert; their id is -1."""
    _C.require_cuda(logits, correction)
    n = experts + identity
    if logits.dtype != torch.float32 or logits.stride(1) != 1 or logits.shape[1] < n:
        raise ValueError("logits must be float32 with dense rows, one column per expert and identity expert")
    if correction is not None and (correction.dtype != torch.float32 or correction.numel() != n or not correction.is_contiguous()):
        raise ValueError(f"correction must be contiguous float32 ({n},)")
    t = logits.shape[0]
    ids = torch.empty((t, top), dtype=torch.int32, device=logits.device)
    weights = torch.empty((t, top), dtype=torch.float32, device=logits.device)
    st = _C.load().mvllm_moe_route_softmax(_ptr(ids), _ptr(weights), _ptr(logits), logits.stride(0) if t > 1 else logits.shape[1],
                                           _ptr(correction), t, experts, identity, top, int(renormalize), _C.current_stream_ptr(logits.device))
    _C.check(st, "moe_route_softmax")
    return ids, weights


def moe_plan(ids: torch.Tensor, experts: int) -> ExpertPlan:
    _C.require_cuda(ids)
    if ids.dtype != torch.int32 or not ids.is_contiguous():
        raise ValueError("ids must be contiguous int32")
    return ExpertPlan(ids, experts)


def moe_linear(x: torch.Tensor, weight: torch.Tensor, ids: torch.Tensor, plan: ExpertPlan | None = None, per_token: int = 0,
               glu: bool | tuple = False, shared: tuple | None = None):
    """Row p = x[row of p] W_e^T for every (token, choice) pair of ``ids`` (T, top), e its expert; with ``glu`` silu(gate) * up, with
    ``glu`` = (alpha, limit, shift) the clamped form of ``layers.fused.gated_unit``.  Pairs with negative ids have no row.

    With a plan rows are in its sorted order, without in the pairs'.  ``per_token`` > 0: pair p reads row p / per_token of x,
    0: row p of x is row p's own (an earlier product's).  weight (E, N, K), with ``glu`` as ``interleave_gate_up`` makes it.

    ``shared``: (x, weight (N, K)) of an expert that all rows go through (bf16, with a plan; with ``glu`` True all gate rows before the up rows), in the same launch;
    the result is then a pair."""
    _C.require_cuda(x, weight, ids)
    experts, n, k = weight.shape
    pairs = ids.numel()
    if x.dim() != 2 or x.shape[1] != k or x.stride(1) != 1 or weight.dtype != x.dtype or not weight.is_contiguous():
        raise ValueError(f"x (*, {k}) with dense rows and a contiguous weight of its dtype expected")
    if ids.dtype != torch.int32 or not ids.is_contiguous() or x.shape[0] * max(per_token, 1) != pairs:
        raise ValueError("ids must be contiguous int32 and x have a row for every token or pair")
    if plan is not None and plan.pairs != pairs:
        raise ValueError("the plan is of other ids")
    out = torch.empty((pairs, n // 2 if glu else n), dtype=x.dtype, device=x.device)
    head = (_ptr(out), out.shape[1], _ptr(x), x.stride(0) if x.shape[0] > 1 else k, _ptr(weight), _ptr(ids),
            _ptr(plan.data if plan is not None else None), pairs, experts, n, k, per_token)
    tail = (_C.dtype_code(x.dtype), _C.current_stream_ptr(x.device))
    if shared is not None:
        xs, ws = shared
        _C.require_cuda(xs, ws)
        if (plan is None or isinstance(glu, tuple) or xs.dim() != 2 or ws.dim() != 2 or xs.shape[1] != ws.shape[1] or xs.stride(1) != 1 or xs.dtype != x.dtype
                or ws.dtype != x.dtype or not ws.is_contiguous()):
            raise ValueError("the shared product takes x (T, K) with dense rows and a contiguous weight (N, K) of the experts' dtype, a plan and no clamped gate")
        t, (m, ks) = xs.shape[0], ws.shape
        beside = torch.empty((t, m // 2 if glu else m), dtype=x.dtype, device=x.device)
        st = _C.load().mvllm_moe_linear_shared(*head, int(glu), _ptr(beside), beside.shape[1], _ptr(xs), xs.stride(0) if t > 1 else ks, _ptr(ws), t, m, ks, *tail)
        _C.check(st, "moe_linear")
        return out, beside
    if isinstance(glu, tuple):
        st = _C.load().mvllm_moe_linear_clamped(*head, *(float(c) for c in glu), *tail)
    else:
        st = _C.load().mvllm_moe_linear(*head, int(glu), *tail)
    _C.check(st, "moe_linear")
    return out


def moe_linear_tiles(pairs: int, experts: int, n: int, k: int, shared: tuple | None = None) -> tuple:
    """(rows, weight rows) of the tiles that a bf16 ``moe_linear`` of these sizes runs on with a plan, ``shared`` = (rows, N, K); host arithmetic only."""
    out = [ctypes.c_int(0), ctypes.c_int(0)]
    st = _C.load().mvllm_moe_linear_tiles(pairs, experts, n, k, *(shared or (0, 0, 0)), *(ctypes.byref(v) for v in out))
    _C.check(st, "moe_linear_tiles")
    return tuple(v.value for v in out)


def interleave_gate_up(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """(F, K) gate and up rows in turns of 32, F a multiple of 32."""
    f, k = gate.shape
    return torch.stack([gate.view(f // 32, 32, k), up.view(f // 32, 32, k)], dim=1).reshape(2 * f, k)


class SparseExperts(nn.Module):
    """``experts`` feed-forwards silu(gate) * up of size ``ff``, ``top`` of them per token, and optionally a shared one behind
    a gate of one number per token.  Inputs are ``inputs`` wide (zeros past the model's width).

    ``softmax``: scores are a softmax over experts and ``identity`` further ones that hand their input on, and weights stay as
    they are; otherwise sigmoids, weights normalized.  ``glu``: (alpha, limit, shift) of clamped gated units."""

    ALIGN = 64             # the products' step along K

    def __init__(self, width: int, inputs: int, experts: int, top: int, ff: int, groups: int = 1, keep: int = 1,
                 shared_ff: int = 0, shared_gate: bool = True, small_rows: int = 0, softmax: bool = False, identity: int = 0,
                 glu: tuple | None = None):
        super().__init__()
        if identity and not softmax:
            raise ValueError("identity experts take a softmax router")
        self.softmax, self.identity, self.glu = softmax, identity, glu if glu is not None else True
        self.width, self.inputs, self.experts, self.top, self.groups, self.keep = width, inputs, experts, top, groups, keep
        self.ff = round_up(ff, self.ALIGN)
        self.shared_gate = shared_gate and shared_ff > 0
        self.shared_ff = round_up(shared_ff, 16) if shared_ff else 0
        if shared_ff:
            with torch.device("meta"):
                self.shared = Qwen3MLP(inputs, self.shared_ff, False, True, small_rows)
        else:
            self.shared = None
        self.correction = None

    @torch.no_grad()
    def load(self, get, matrix):
        """``get(name)``: checkpoint tensor, ``matrix(t)``: a product's weight on the device in the model's type."""
        def expert(e):
            gate, up = (pad_to(matrix(get(f"e{e}.{n}")), self.ff, self.inputs) for n in ("gate", "up"))
            return interleave_gate_up(gate, up), pad_to(matrix(get(f"e{e}.down")), round_up(self.width, 16), self.ff)

        first = expert(0)
        self.gate_up = first[0].new_empty((self.experts, *first[0].shape))
        self.down = first[1].new_empty((self.experts, *first[1].shape))
        for e in range(self.experts):
            self.gate_up[e], self.down[e] = first if e == 0 else expert(e)
        rows = [get("router")] + ([get("shared.sg")] if self.shared_gate else [])
        self.router = pad_to(torch.cat([matrix(r) for r in rows]), None, self.inputs)
        self.correction = get("correction").to(device=self.router.device, dtype=torch.float32).contiguous()
        if self.shared is not None:
            gate, up = (pad_to(matrix(get(f"shared.{n}")), self.shared_ff, self.inputs) for n in ("gate", "up"))
            self.shared.gate_up.weight = nn.Parameter(torch.cat([gate, up]), requires_grad=False)
            self.shared.gate_down.weight = nn.Parameter(pad_to(matrix(get("shared.down")), None, self.shared_ff), requires_grad=False)

    def _shared_beside(self, h) -> bool:
        """Whether the shared expert's products may be part of the experts' launches: not where it is not as built here, somebody hooked into it, or the
        launches do not take its sizes."""
        m = self.shared
        if (m is None or self.glu is not True or h.dtype != torch.bfloat16 or h.dim() != 2 or h.shape[0] == 0 or not self._beside_pays(h.shape[0])
                or _has_any_global_hook() or not _as_built(m, Qwen3MLP)):
            return False
        gate_up, gate_down = m.gate_up, m.gate_down
        if not _as_built(gate_up, Linear) or not _as_built(gate_down, Linear) or not _as_built(m.activation, SiluAndMul):
            return False
        up, down = gate_up.weight, gate_down.weight
        if torch.is_grad_enabled() and (h.requires_grad or up.requires_grad or down.requires_grad):
            return False
        # (a weight of a class of its own may hold other numbers than its memory, as quantized ones do)
        if type(up) not in _PLAIN or type(down) not in _PLAIN or gate_up.bias is not None or gate_down.bias is not None:
            return False
        (rows, inputs), (n, k), (width, ff) = h.shape, up.shape, down.shape
        return (up.dtype == down.dtype == h.dtype and up.device == down.device == h.device and up.is_contiguous() and down.is_contiguous()
                and n == 2 * ff and k == inputs and ff % 64 == 0 and width % 16 == 0 and up.data_ptr() % 16 == 0 and down.data_ptr() % 16 == 0
                # offsets of 32 bits into weights and, unsigned, rows
                and n * k < 1 << 30 and width * ff < 1 << 30 and _span(h) < 1 << 31 and rows * ff < 1 << 31)

    def _beside_pays(self, rows: int) -> bool:
        """Whether the shared expert's products are better off in the experts' launches.

        They run on tiles made for the experts' rows.  The few long tiles (K of ``shared_ff``) of a shared expert that is large, and much larger than the others, are
        still running when all others are done, unless large tiles share the rounds out; and tiles of 64 rows (``rows * top`` up to 48 per expert) are far
        behind the library's product once there are many.  785 mixtures of 8 to 256 experts of 64 to 2048, shared ones of 64 to 10240, 1 to 8192 rows:
        within these lines 1.14 times as fast on average, 8 of 600 more than 3 % slower (worst 0.914); beyond them 0.99, 69 of 185 more than 3 % slower (worst
        0.63).  us apart / beside, 2048 wide: 8 experts of 1408 and 7680 shared, 56 rows 83 / 114; top 1 of 64 of 1536 and 8448, 2627 rows 552 / 761; top 1 of
        256 of 704 and 1344, 7911 rows 540 / 626.  From 96 rows per expert on a large shared expert is as well off: top 4 of 64 of 1408 and 5632, 2048 rows
        498 / 443."""
        pairs = rows * self.top
        return (self.shared_ff <= max(2048, 3.5 * self.ff) or pairs >= 96 * self.experts) and (rows <= 1500 or pairs > 48 * self.experts)

    def _sorted(self, h, pairs: int, beside: bool) -> bool:
        """Whether the products go over sorted pairs: always but for few pairs in 16 bits, and for those too where it pays (``SHORT_ROWS``) and offsets into an
        expert's weights and the rows are of 32 bits."""
        if h.dtype != torch.bfloat16 or pairs > FEW_PAIRS:
            return True
        return (pairs > 0 and (beside or max(self.inputs, self.ff) >= SHORT_ROWS) and 4 * self.ff * self.inputs < 1 << 31 and _span(h) < 1 << 31)

    def forward(self, h) -> ExpertOutput:
        logits = gate_linear(h, self.router, None, self.router.shape[0], 0.0)
        if self.softmax:
            ids, weights = moe_route_softmax(logits, self.correction, self.experts, self.identity, self.top)
        else:
            ids, weights = moe_route(logits, self.correction, self.experts, self.top, self.groups, self.keep)
        pairs = ids.numel()
        plan = None
        beside = self._shared_beside(h)
        if self._sorted(h, pairs, beside):
            plan = moe_plan(ids, self.experts)
        shared = None
        if plan is not None and beside:
            act, shared = moe_linear(h, self.gate_up, ids, plan, self.top, glu=True, shared=(h, self.shared.gate_up.weight))
            parts, shared = moe_linear(act, self.down, ids, plan, shared=(shared, self.shared.gate_down.weight))
        else:
            act = moe_linear(h, self.gate_up, ids, plan, self.top, glu=self.glu)
            parts = moe_linear(act, self.down, ids, plan)
        out = ExpertOutput(parts, weights, None if plan is None else plan.place)
        if self.identity:
            out.ids, out.inputs = ids, h
        if self.shared is not None:
            out.shared = self.shared(h) if shared is None else shared
            out.gate = logits[:, self.experts] if self.shared_gate else None
        return out
