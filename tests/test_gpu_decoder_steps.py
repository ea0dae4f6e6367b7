"""The decoder's layers at a decode step's rows, with norms as part of the projections before or behind them, against the chain of separate modules.

Both are the same 16-bit network, rounded at the same places, and differ from it in fp32 by those roundings; sums in another order make single roundings
fall the other way, which moves that difference by a fraction of itself, while a residual or a norm that is not the right one is an error of the values' own size."""
import pytest
import torch
import torch.nn as nn

import minivllm_amd.models.qwen3 as qwen3
from minivllm_amd.models.qwen3 import Qwen3ForCausalLM

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
HEADS, GROUPS, LAYERS = 16, 8, 3


class MeanOfValues(nn.Module):
    """In the attention operator's place: something of q, k and v."""

    def forward(self, q, k, v):
        return (0.5 * q + 0.5 * (k + v).repeat_interleave(q.shape[1] // k.shape[1], 1)).flatten(1)


def decoder(width, ff, heads, dtype, small_rows, **kw):
    model = Qwen3ForCausalLM(512, width, heads, head_dim=128, num_kv_heads=GROUPS, intermediate_size=ff, num_layers=LAYERS, fused_qk=False, ffn_bias=True, max_position=256,
                             fused_elementwise=small_rows > 0, small_rows=small_rows, **kw)
    model.reset_parameters(seed=1, std=0.04)
    for i, p in enumerate(model.parameters()):
        if p.dim() == 1:
            p.data += 0.2 * torch.randn(p.shape, generator=torch.Generator().manual_seed(i))
        p.data = p.data.bfloat16().float()                        # the same numbers in every dtype
    for layer in model.layer_stack:
        layer.self_attn.attention = MeanOfValues()
    return model.to(dtype).to(DEV).requires_grad_(False)


# (output projections, down projections) that take the norm behind them, of LAYERS each; the last down projection has the final norm
@pytest.mark.parametrize("width,ff,heads,rows,outs,downs", [
    (1024, 3072, HEADS, 3, 0, 0), (1024, 3072, HEADS, 4, 0, 1), (1024, 3072, HEADS, 16, 0, 1),         # both norms in the products behind them
    (1024, 3072, HEADS, 17, 3, 3), (1024, 3072, HEADS, 61, 3, 3), (1024, 3072, HEADS, 64, 3, 3), (1024, 3072, HEADS, 65, 0, 0),
    (1024, 6144, HEADS, 5, 3, 1), (1024, 6144, HEADS, 16, 3, 1),      # gate and up are too wide for it: output projections, and the last down projection
    (1024, 3072, 64, 5, 0, 3), (1024, 3072, 64, 16, 0, 3),            # q, k and v are: down projections
    (2048, 6144, HEADS, 3, 0, 0), (2048, 6144, HEADS, 4, 3, 3), (2048, 6144, HEADS, 16, 3, 3), (2048, 6144, HEADS, 17, 3, 3), (2048, 6144, HEADS, 61, 3, 3)])
def test_steps_with_joined_norms(monkeypatch, width, ff, heads, rows, outs, downs):
    ran = []
    join = qwen3.linear_add_rms_norm
    monkeypatch.setattr(qwen3, "linear_add_rms_norm", lambda x, *more: (ran.append(x.shape[1]), join(x, *more))[1])
    ids, at = torch.arange(rows, device=DEV) * 7 % 512, torch.arange(rows, device=DEV)
    got = decoder(width, ff, heads, torch.bfloat16, 64)(ids, at).float()
    assert (ran.count(heads * 128), ran.count(ff)) == (outs, downs), ran
    chain = decoder(width, ff, heads, torch.bfloat16, 0)(ids, at).float()
    assert len(ran) == outs + downs
    exact = decoder(width, ff, heads, torch.float32, 0)(ids, at)
    off, usual = ((x - exact).norm().item() / exact.norm().item() for x in (got, chain))
    assert usual < 0.05 and off < 1.3 * usual, (off, usual)
