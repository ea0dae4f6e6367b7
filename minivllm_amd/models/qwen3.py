"""Qwen3-style decoder used as the caller of the attention path (src/myvllm/models/qwen3.py).

Single-GPU PyTorch-ROCm: the projections are plain ``F.linear`` (hipBLASLt); the only custom kernels
are behind ``minivllm_amd.layers.attention.Attention``.  Shapes follow the intended semantics where the
reference's own do not work: the QKV projection maps ``hidden_size`` (not ``num_heads*head_dim``,
qwen3.py:37-43) to ``(Hq + 2 Hkv) * D``; ``rms_norm_epsilon`` is honoured (the reference accepts and drops
it); ``Attention`` receives the engine's ``block_size``; weights are seeded N(0, 0.02) instead of
uninitialised memory.  Positions are computed once per step by the model runner, not per layer.
"""
from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.nn.modules.module import _has_any_global_hook

from minivllm_amd.layers.attention import Attention
from minivllm_amd.layers.basic import Linear, RMSNorm, RotaryEmbedding, SiluAndMul
from minivllm_amd.layers.fused import linear_add_rms_norm, linear_add_rms_norm_takes, norm_linear_small_m, norm_linear_small_m_pays, norm_linear_small_m_takes
from minivllm_amd.utils.context import get_context


def _as_built(module, kind):
    """Whether calling ``module`` is ``kind.forward`` and nothing else, so that its work may be done as a part of another launch: not where it was
    replaced, or somebody hooked into it (hooks on all modules: ``_has_any_global_hook``).  A step asks this of every module it passes by: 0.3 us each."""
    own = module.__dict__
    return type(module) is kind and not (own["_forward_hooks"] or own["_forward_pre_hooks"] or "forward" in own)


# a norm between two projections: nobody has looked yet, it has been applied with the one before, it is to run in the one behind
_OPEN, _NORMED, _INSIDE = range(3)


class Qwen3Attention(nn.Module):
    def __init__(self, hidden_size, num_heads, head_dim, scale, num_kv_heads, rms_norm_epsilon, qkv_bias,
                 rotary: RotaryEmbedding, block_size, kv_cache_dtype, fused_qk=True, small_rows=0):
        super().__init__()
        self.num_heads, self.num_kv_heads, self.head_dim = num_heads, num_kv_heads, head_dim
        self.q_size, self.kv_size = num_heads * head_dim, num_kv_heads * head_dim
        self.qkv_projection = Linear(hidden_size, self.q_size + 2 * self.kv_size, bias=qkv_bias, small_rows=small_rows)
        self.qkv_bias = qkv_bias
        self.rms_norm = RMSNorm(head_dim, rms_norm_epsilon)      # one gamma shared by q and k (qwen3.py:50, 104-106)
        self.rotary_emb = rotary
        self.attention = Attention(num_heads, head_dim, scale, num_kv_heads, block_size, kv_cache_dtype)
        self.output_projection = Linear(self.q_size, hidden_size, bias=False, small_rows=small_rows)
        self.fused_qk = fused_qk

    def forward(self, x, positions):
        return self.forward_qkv(self.qkv_projection(x), positions)

    def forward_qkv(self, qkv, positions):
        """Everything after the QKV projection (whose output a caller may have produced fused with the norm)."""
        return self.output_projection(self.attend(qkv, positions))

    def attend(self, qkv, positions):
        """``forward_qkv`` without the output projection."""
        q, k, v = qkv.split([self.q_size, self.kv_size, self.kv_size], dim=-1)
        if self.fused_qk:
            # views of the projection output, no copies; norm + rotation + cache store in one launch
            q = q.unflatten(-1, (self.num_heads, self.head_dim))
            k = k.unflatten(-1, (self.num_kv_heads, self.head_dim))
            v = v.unflatten(-1, (self.num_kv_heads, self.head_dim))
            gamma = None if self.qkv_bias else self.rms_norm.weight_fp32()
            return self.attention.forward_fused(q, k, v, positions, self.rotary_emb.cos_sin_cache, gamma,
                                                self.rms_norm.eps)
        q = q.reshape(-1, self.num_heads, self.head_dim)
        k = k.reshape(-1, self.num_kv_heads, self.head_dim)
        v = v.reshape(-1, self.num_kv_heads, self.head_dim)
        if not self.qkv_bias:
            q, k = self.rms_norm(q), self.rms_norm(k)
        q, k = self.rotary_emb(positions, q, k)
        return self.attention(q, k, v)


class Qwen3MLP(nn.Module):
    def __init__(self, hidden_size, intermediate_size, bias, fused=True, small_rows=0):
        super().__init__()
        self.gate_up = Linear(hidden_size, 2 * intermediate_size, bias=bias, small_rows=small_rows)
        self.activation = SiluAndMul(fused)
        self.gate_down = Linear(intermediate_size, hidden_size, bias=bias, small_rows=small_rows)
        self.small_rows, self.fused = small_rows, fused

    def forward(self, x):
        return self.gate_down(self.gated(x))

    def gated(self, x):
        """``forward`` without the last projection."""
        # a decode step's rows: SiluAndMul as the epilogue of the gate/up projection (one launch instead of two)
        if (self.small_rows and self.fused and x.dim() == 2 and x.shape[0] <= self.small_rows and x.is_contiguous()
                and _as_built(self.gate_up, Linear) and _as_built(self.activation, SiluAndMul) and not _has_any_global_hook()
                and norm_linear_small_m_takes(x, self.gate_up.weight, self.small_rows, norm=False, glu=True)):
            return norm_linear_small_m(x, self.gate_up.weight, self.gate_up.bias, glu=True)
        return self.activation(self.gate_up(x))


class Qwen3DecoderLayer(nn.Module):
    def __init__(self, hidden_size, intermediate_size, ffn_bias, rms_norm_epsilon, fused_elementwise=True,
                 small_rows=0, norm_rows=32, **attn_kwargs):
        super().__init__()
        self.input_layernorm = RMSNorm(hidden_size, rms_norm_epsilon, fused_elementwise)
        self.self_attn = Qwen3Attention(hidden_size=hidden_size, rms_norm_epsilon=rms_norm_epsilon,
                                        small_rows=small_rows, **attn_kwargs)
        self.post_attention_layernorm = RMSNorm(hidden_size, rms_norm_epsilon, fused_elementwise)
        self.mlp = Qwen3MLP(hidden_size, intermediate_size, ffn_bias, fused_elementwise, small_rows)
        self.norm_rows, self.fused_elementwise = min(small_rows, norm_rows), fused_elementwise

    def _norm_in_product(self, norm, proj, x, glu=False, joins=False):
        """A decode step's few rows: the residual norm runs as the prologue of the projection behind it (and SiluAndMul as its
        epilogue) where that is faster than a launch of its own or, with ``joins``, than as part of the projection before it; the roundings are the same."""
        if not (self.norm_rows and self.fused_elementwise and x.dim() == 2 and x.shape[0] <= self.norm_rows and x.is_contiguous()
                and _as_built(norm, RMSNorm) and _as_built(proj, Linear)):
            return False
        weight = proj.weight
        return norm_linear_small_m_pays(x.shape[0], weight, joins) and norm_linear_small_m_takes(x, weight, self.norm_rows, glu=glu)

    def _project_norm(self, proj, x, residual, norm, into, glu=False):
        """``norm(proj(x), residual)`` where the norm can join the projection and is not better off in ``into``, the projection behind it (None: unknown),
        else the projection and ``residual`` as it is; and which."""
        if norm is None or not _as_built(proj, Linear):
            return proj(x), residual, _OPEN
        if into is not None and self._norm_in_product(norm, into, residual, glu, joins=True):
            return proj(x), residual, _INSIDE
        if (self.norm_rows and proj.small_rows and norm.fused and _as_built(norm, RMSNorm)
                and linear_add_rms_norm_takes(x, proj.weight, residual, proj.small_rows)):
            return *linear_add_rms_norm(x, proj.weight, proj.bias, residual, norm.weight_fp32(), norm.eps), _NORMED
        return proj(x), residual, _OPEN

    def forward(self, x, residual, positions):
        return self.walk(x, residual, positions)[:2]

    def walk(self, x, residual, positions, state=_OPEN, behind=None, into=None):
        """``forward`` for a caller that knows its neighbours: ``state`` of the input norm; ``behind``, the norm that follows the
        layer and may be applied here, with ``into`` the projection that follows it.  The third result is that norm's state.  Modules that are not as
        this file builds them are called as they are."""
        attn, mlp, norm = self.self_attn, self.mlp, self.input_layernorm
        free = not _has_any_global_hook()
        own_attn = free and _as_built(attn, Qwen3Attention)
        own_mlp = free and _as_built(mlp, Qwen3MLP) and _as_built(mlp.activation, SiluAndMul)
        qkv = None
        if state == _NORMED:
            pass
        elif own_attn and (state == _INSIDE or self._norm_in_product(norm, attn.qkv_projection, x)):
            proj = attn.qkv_projection
            qkv = norm_linear_small_m(x, proj.weight, proj.bias, norm.weight_fp32(), norm.eps, residual, residual is not None)
            qkv, residual = (qkv, x) if residual is None else qkv
        elif residual is None:
            residual, x = x, norm(x)
        else:
            x, residual = norm(x, residual)
        norm, state = self.post_attention_layernorm, _OPEN
        if own_attn:
            x = attn.attend(attn.qkv_projection(x) if qkv is None else qkv, positions)
            x, residual, state = self._project_norm(attn.output_projection, x, residual, norm, mlp.gate_up if own_mlp else None, glu=True)
        else:
            x = attn(x, positions)
        if state != _NORMED and own_mlp and (state == _INSIDE or self._norm_in_product(norm, mlp.gate_up, x, glu=True)):
            proj = mlp.gate_up
            x, residual = norm_linear_small_m(x, proj.weight, proj.bias, norm.weight_fp32(), norm.eps, residual, True, glu=True)
        else:
            if state != _NORMED:
                x, residual = norm(x, residual)
            if not own_mlp:
                return mlp(x), residual, _OPEN
            x = mlp.gated(x)
        return self._project_norm(mlp.gate_down, x, residual, behind, into)


class Qwen3ForCausalLM(nn.Module):
    def __init__(self, vocab_size, hidden_size, num_heads, head_dim=None, scale=1.0, num_kv_heads=None,
                 rms_norm_epsilon=1e-6, qkv_bias=False, base=1_000_000, max_position=4096,
                 intermediate_size=3072, ffn_bias=True, num_layers=8, tie_word_embeddings=True,
                 block_size=256, kv_cache_dtype="auto", fused_qk=True, fused_elementwise=True, small_rows=0,
                 norm_rows=32):
        super().__init__()
        head_dim = head_dim if head_dim is not None else hidden_size // num_heads
        num_kv_heads = num_kv_heads if num_kv_heads is not None else num_heads
        self.embedding_layer = nn.Embedding(vocab_size, hidden_size)
        rotary = RotaryEmbedding(base, head_dim, max_position)
        self.layer_stack = nn.ModuleList([
            Qwen3DecoderLayer(hidden_size, intermediate_size, ffn_bias, rms_norm_epsilon, num_heads=num_heads,
                              head_dim=head_dim, scale=scale, num_kv_heads=num_kv_heads, qkv_bias=qkv_bias,
                              rotary=rotary, block_size=block_size, kv_cache_dtype=kv_cache_dtype,
                              fused_qk=fused_qk, fused_elementwise=fused_elementwise, small_rows=small_rows,
                              norm_rows=norm_rows)
            for _ in range(num_layers)])
        self.final_layernorm = RMSNorm(hidden_size, rms_norm_epsilon, fused_elementwise)
        self.lm_head_weight = self.embedding_layer.weight if tie_word_embeddings else nn.Parameter(
            torch.empty(vocab_size, hidden_size))
        self.max_position = max_position

    def reset_parameters(self, seed: int = 0, std: float = 0.02):
        g = torch.Generator(device="cpu").manual_seed(seed)
        with torch.no_grad():
            for name, p in self.named_parameters():
                if p.dim() >= 2:
                    p.copy_(torch.randn(p.shape, generator=g) * std)
                elif name.endswith("bias"):
                    p.zero_()
                else:
                    p.fill_(1.0)

    def forward(self, input_ids, positions):
        # a decode step's few rows by plain indexing: the embedding operator's small-batch kernel takes 11 us for 16
        # rows, the gather 4
        x = self.embedding_layer.weight[input_ids] if input_ids.numel() <= 256 else self.embedding_layer(input_ids)
        residual, state, layers = None, _OPEN, list(self.layer_stack)
        free = not _has_any_global_hook()
        own = [free and _as_built(layer, Qwen3DecoderLayer) for layer in layers]
        for i, layer in enumerate(layers):
            behind = into = None
            if i + 1 == len(layers):
                behind = self.final_layernorm if free else None
            elif own[i + 1]:
                behind, attn = layers[i + 1].input_layernorm, layers[i + 1].self_attn
                into = attn.qkv_projection if _as_built(attn, Qwen3Attention) else None
            if own[i]:
                x, residual, state = layer.walk(x, residual, positions, state, behind, into)
            else:
                x, residual = layer(x, residual, positions)
                state = _OPEN
        return x if state == _NORMED else self.final_layernorm(x, residual)[0]

    def compute_logits(self, hidden):
        context = get_context()
        if context.is_prefill:                         # last token of every packed sequence (embedding_head.py:57-62)
            hidden = hidden[(context.cu_seqlens_q[1:] - 1).long()].contiguous()
        return F.linear(hidden, self.lm_head_weight)
