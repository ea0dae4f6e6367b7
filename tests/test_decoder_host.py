"""The decoder's steps of few rows, where norms join the projections around them: the wiring, with the launches as tensor operations.  A module that
was replaced or hooked into has to be called, at every number of rows."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

import minivllm_amd.layers.basic as basic
import minivllm_amd.models.qwen3 as qwen3
from minivllm_amd.layers.basic import Linear
from minivllm_amd.layers.fused import norm_linear_small_m_pays
from minivllm_amd.models.qwen3 import Qwen3DecoderLayer, Qwen3ForCausalLM


class MeanOfValues(nn.Module):
    """In the attention operator's place: something of q, k and v."""

    def forward(self, q, k, v):
        return (q + (k + v).repeat_interleave(q.shape[1] // k.shape[1], 1)).flatten(1)


def norm_of(x, gamma, eps):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps) * gamma


def add_rms_norm(x, gamma, eps, residual=None):
    return norm_of(x, gamma, eps) if residual is None else (norm_of(x + residual, gamma, eps), x + residual)


def gated(x):
    a, b = x.chunk(2, -1)
    return F.silu(a) * b


@pytest.fixture
def joined(monkeypatch):
    """The launches as tensor operations; which of them ran.  Few rows in the product behind the norm, more in the one before."""
    calls = []

    def join(x, weight, bias, residual, gamma, eps):
        calls.append("join")
        h = F.linear(x, weight, bias) + residual
        return norm_of(h, gamma, eps), h

    def prologue(x, weight, bias=None, gamma=None, eps=1e-6, residual=None, want_residual=False, glu=False):
        calls.append("prologue" if gamma is not None else "glu")
        h = x if residual is None else x + residual
        y = F.linear(h if gamma is None else norm_of(h, gamma, eps), weight, bias)
        y = gated(y) if glu else y
        return (y, h) if want_residual else y

    monkeypatch.setattr(basic, "add_rms_norm", add_rms_norm)
    monkeypatch.setattr(basic, "silu_and_mul", gated)
    monkeypatch.setattr(qwen3, "linear_add_rms_norm", join)
    monkeypatch.setattr(qwen3, "norm_linear_small_m", prologue)
    monkeypatch.setattr(qwen3, "linear_add_rms_norm_takes", lambda x, w, r, most=64: 4 <= x.shape[0] <= most and r.shape == (x.shape[0], w.shape[0]))
    monkeypatch.setattr(qwen3, "norm_linear_small_m_takes", lambda x, w, most=64, norm=True, glu=False: x.shape[0] <= most)
    monkeypatch.setattr(qwen3, "norm_linear_small_m_pays", lambda rows, w, *more: rows <= 6)
    return calls


def decoder(**kw):
    model = Qwen3ForCausalLM(64, 32, 4, head_dim=8, num_kv_heads=2, intermediate_size=48, num_layers=3, fused_qk=False, ffn_bias=True, max_position=128, small_rows=64, **kw)
    model.reset_parameters(seed=3, std=0.3)
    for i, p in enumerate(model.parameters()):
        if p.dim() == 1:
            p.data += 0.1 * torch.randn(p.shape, generator=torch.Generator().manual_seed(i))
    for layer in model.layer_stack:
        layer.self_attn.attention = MeanOfValues()
    return model.double().requires_grad_(False)


def expected(model, ids):
    """The decoder as its modules say, one after the other."""
    x, residual = model.embedding_layer.weight[ids], None
    at = torch.arange(len(ids))
    for layer in model.layer_stack:
        if type(layer) is not Qwen3DecoderLayer:
            x, residual = layer(x, residual, at)
            continue
        h = x if residual is None else x + residual
        x = layer.self_attn(layer.input_layernorm(h), at)
        h = x + h
        x, residual = layer.mlp(layer.post_attention_layernorm(h)), h
        for hook in layer._forward_hooks.values():
            x, residual = hook(layer, None, (x, residual))
    return model.final_layernorm(x + residual)


@pytest.mark.parametrize("rows", [1, 3, 4, 6, 7, 64, 65])
def test_steps_are_the_chain_of_modules(joined, rows):
    model, ids = decoder(), torch.arange(rows) % 64
    got, ran = model(ids, torch.arange(rows)), set(joined)
    assert ran == ({"prologue", "join"} if 4 <= rows <= 6 else {"prologue"} if rows < 4 else {"join", "glu"} if rows <= 64 else set())
    assert torch.allclose(got, expected(model, ids), rtol=1e-4, atol=1e-4)       # (gamma in fp32)


@pytest.mark.parametrize("rows,prologues,joins", [(3, 6, 0), (4, 1, 6), (16, 1, 6), (17, 0, 6)])
def test_a_norm_without_a_projection_before_it(joined, monkeypatch, rows, prologues, joins):
    """Long rows: the norms join the projections before them from 4 rows on.  The first has none and stays in the product behind it up to 16."""
    monkeypatch.setattr(qwen3, "norm_linear_small_m_pays", lambda rows, w, joins=False: norm_linear_small_m_pays(rows, torch.empty(4096, 2048, device="meta"), joins))
    model, ids = decoder(), torch.arange(rows)
    got = model(ids, ids)
    assert (joined.count("prologue"), joined.count("join")) == (prologues, joins) and torch.allclose(got, expected(model, ids), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("n,k,rows,joins,pays", [(4096, 1024, 16, True, True), (4096, 1024, 17, True, False), (4096, 2048, 3, True, True), (4096, 2048, 4, True, False),
                                                 (4096, 2048, 16, False, True), (4096, 2048, 17, False, False), (4112, 2048, 1, False, False)])
def test_norm_in_product_rule(n, k, rows, joins, pays):
    assert norm_linear_small_m_pays(rows, torch.empty(n, k, device="meta"), joins) == pays


@pytest.mark.parametrize("rows", [2, 5, 30, 64])
def test_no_norm_rows_no_joined_norms(joined, rows):
    model, ids = decoder(norm_rows=0), torch.arange(rows)
    got = model(ids, ids)
    assert set(joined) == {"glu"} and torch.allclose(got, expected(model, ids), rtol=1e-4, atol=1e-4)


def double(module, args, out):
    return 2 * out


class Shifted(nn.Module):
    """A module of another kind around the built one."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, *args):
        return self.inner(*args) + 0.5


class OwnLayer(nn.Module):
    def forward(self, x, residual, positions):
        return torch.tanh(x), x if residual is None else residual - x


def hook(path):
    return lambda model: model.get_submodule(path).register_forward_hook(double)


def pre_hook(path):
    return lambda model: model.get_submodule(path).register_forward_pre_hook(lambda module, args: (args[0] * 3, *args[1:]))


def replace(path):
    parent, _, name = path.rpartition(".")
    return lambda model: setattr(model.get_submodule(parent), name, Shifted(model.get_submodule(path)))


def plain_linear(path):
    parent, _, name = path.rpartition(".")

    def change(model):
        old = model.get_submodule(path)
        new = nn.Linear(old.in_features, old.out_features, old.bias is not None).double().requires_grad_(False)
        new.load_state_dict(old.state_dict())
        new.weight *= 2
        setattr(model.get_submodule(parent), name, new)
    return change


def own_forward(path):
    def change(model):
        module = model.get_submodule(path)
        was = module.forward
        module.forward = lambda *args: 2 * was(*args)
    return change


def own_layer(model):
    model.layer_stack[1] = OwnLayer()


def layer_hook(model):
    # right for what a layer returns: an output and a residual that are added by whatever follows
    model.layer_stack[1].register_forward_hook(lambda layer, args, out: (0.5 * (out[0] + out[1]), 0.5 * (out[0] + out[1])))


CHANGES = {**{f"hook {p}": hook(p) for p in ("layer_stack.1.mlp.gate_down", "layer_stack.0.mlp", "layer_stack.1.self_attn", "layer_stack.1.self_attn.output_projection",
                                            "layer_stack.2.self_attn.qkv_projection", "layer_stack.1.mlp.gate_up", "layer_stack.0.mlp.activation")},
           **{f"pre-hook {p}": pre_hook(p) for p in ("layer_stack.1.mlp.gate_down", "layer_stack.1.self_attn.output_projection", "layer_stack.1.mlp")},
           **{f"replaced {p}": replace(p) for p in ("layer_stack.1.mlp.gate_down", "layer_stack.0.self_attn", "layer_stack.2.mlp", "layer_stack.1.self_attn.output_projection",
                                                    "layer_stack.0.self_attn.qkv_projection", "layer_stack.2.mlp.gate_up")},
           **{f"nn.Linear {p}": plain_linear(p) for p in ("layer_stack.1.mlp.gate_down", "layer_stack.1.self_attn.output_projection", "layer_stack.0.mlp.gate_up")},
           **{f"forward of {p}": own_forward(p) for p in ("layer_stack.1.mlp.gate_down", "layer_stack.2.mlp", "layer_stack.1.self_attn")},
           "own layer": own_layer, "layer's hook": layer_hook}


@pytest.mark.parametrize("rows", [2, 5, 9, 70])
@pytest.mark.parametrize("change", CHANGES)
def test_changed_modules_are_called(joined, change, rows):
    model, ids = decoder(), torch.arange(rows) % 64
    CHANGES[change](model)
    assert torch.allclose(model(ids, torch.arange(rows)), expected(model, ids), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("rows", [2, 5, 9, 70])
@pytest.mark.parametrize("norm", ["layer_stack.1.input_layernorm", "layer_stack.1.post_attention_layernorm", "final_layernorm"])
def test_hooks_on_norms_run(joined, norm, rows):
    model, ids, seen = decoder(), torch.arange(rows) % 64, []
    model.get_submodule(norm).register_forward_hook(lambda module, args, out: seen.append(len(args[0])))
    want = decoder()(ids, torch.arange(rows))
    assert torch.allclose(model(ids, torch.arange(rows)), want, rtol=1e-4, atol=1e-4) and seen == [rows]


def test_hooks_on_every_module_run(joined):
    model, ids, seen = decoder(), torch.arange(9), []
    handle = nn.modules.module.register_module_forward_hook(lambda module, args, out: seen.append(module))
    try:
        model(ids, torch.arange(9))
    finally:
        handle.remove()
    assert sum(isinstance(m, Linear) for m in seen) == 3 * 4 and sum(isinstance(m, Qwen3DecoderLayer) for m in seen) == 3


def test_a_layer_returns_two_values(joined):
    model = decoder()
    x = torch.randn(9, 32, dtype=torch.float64)
    out = model.layer_stack[0](x, None, torch.arange(9))
    assert len(out) == 2
    h = layer_in = x
    layer = model.layer_stack[0]
    h = layer.self_attn(layer.input_layernorm(layer_in), torch.arange(9)) + layer_in
    assert torch.allclose(out[0], layer.mlp(layer.post_attention_layernorm(h)), rtol=1e-4, atol=1e-4) and torch.allclose(out[1], h, rtol=1e-4, atol=1e-4)
