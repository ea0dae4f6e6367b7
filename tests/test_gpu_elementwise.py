"""add_rms_norm and silu_and_mul on the GPU vs the CPU oracle of the reference's tensor-operation chains.

Tolerances.  add_rms_norm: the residual sum is bit-exact; the norm differs from the oracle only through the
order of the sum of squares, so for bf16/fp16 at least 99.5 % of the elements are bit-exact and all are within
1 ulp (2^-7 / 2^-10 relative), fp32 within 2^-19 relative (a sum of up to 8192 squares in another order).  silu_and_mul: exp differs from the CPU's by an ulp or
two of fp32, which the rounding to bf16/fp16 absorbs except at rounding boundaries: same bars, with 2 ulp for
the product (a silu that rounds the other way moves it by one more)."""
import pytest
import torch

import oracle
from minivllm_amd.layers.fused import add_rms_norm, silu_and_mul

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -19}


def _close(got, want, dtype, ulps=1.0):
    got = got.cpu()
    assert got.dtype == dtype and got.shape == want.shape
    if dtype != torch.float32:
        same = (got == want).float().mean().item()
        assert same >= 0.995, f"only {same:.4f} bit-exact"
    err = (got.float() - want.float()).abs()
    assert bool((err <= want.float().abs() * ULP[dtype] * ulps + 1e-30).all()), float(err.max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,hidden", [(64, 1024), (1, 1024), (7, 4096), (3, 8), (5, 520), (2, 8192), (300, 2048)])
@pytest.mark.parametrize("with_residual", [True, False])
def test_add_rms_norm(dtype, rows, hidden, with_residual):
    g = torch.Generator().manual_seed(rows * 31 + hidden)
    x = (torch.randn(rows, hidden, generator=g) * 2).to(dtype)
    r = torch.randn(rows, hidden, generator=g).to(dtype) if with_residual else None
    gamma = torch.rand(hidden, generator=g) + 0.5
    if with_residual:
        want_y, want_s = oracle.add_rms_norm_oracle(x, gamma, 1e-6, r)
        got_y, got_s = add_rms_norm(x.to(DEV), gamma.to(DEV), 1e-6, r.to(DEV))
        assert torch.equal(got_s.cpu().view(torch.uint8), want_s.view(torch.uint8))
    else:
        want_y = oracle.add_rms_norm_oracle(x, gamma, 1e-6)
        got_y = add_rms_norm(x.to(DEV), gamma.to(DEV), 1e-6)
    _close(got_y, want_y, dtype)


@pytest.mark.parametrize("rows", [3071, 3073])
@pytest.mark.parametrize("hidden", [1032, 1088, 1096, 1280, 1288])
@pytest.mark.parametrize("with_residual", [True, False])
def test_add_rms_norm_one_wave_or_four(rows, hidden, with_residual):
    """Both sides of the line between a wave and four per row, a last workgroup that is not full; the last rows against the oracle."""
    g = torch.Generator().manual_seed(rows + hidden)
    x, r = (torch.randn(rows, hidden, generator=g).bfloat16() for _ in range(2))
    gamma = torch.rand(hidden, generator=g) + 0.5
    got = add_rms_norm(x.to(DEV), gamma.to(DEV), 1e-6, r.to(DEV) if with_residual else None)
    want = oracle.add_rms_norm_oracle(x[-70:], gamma, 1e-6, *([r[-70:]] if with_residual else []))
    if with_residual:
        assert torch.equal(got[1].cpu(), (x.float() + r.float()).bfloat16())
        got, want = got[0], want[0]
    _close(got[-70:], want, torch.bfloat16)
    assert torch.isfinite(got).all()


def test_add_rms_norm_more_rows_than_a_launch_counts():
    """2^32 threads and some more: rows on both sides of the end of the first launch, which holds 2^24 - 1 rows of more than 1024 numbers."""
    rows, hidden, first = 2 ** 24 + 2, 1032, 2 ** 24 - 1
    x = torch.empty(rows, hidden, dtype=torch.bfloat16, device=DEV)
    at = torch.tensor([0, first - 1, first, first + 1, rows - 1], device=DEV)
    some = torch.randn(len(at), hidden, generator=torch.Generator().manual_seed(3)).bfloat16()
    x[at], gamma = some.to(DEV), torch.linspace(0.5, 1.5, hidden)
    got = add_rms_norm(x, gamma.to(DEV), 1e-6)[at]
    del x
    torch.cuda.empty_cache()
    _close(got, oracle.add_rms_norm_oracle(some, gamma, 1e-6), torch.bfloat16)


def test_add_rms_norm_strided_rows_and_errors():
    g = torch.Generator().manual_seed(2)
    wide = torch.randn(9, 3 * 512, generator=g).to(torch.bfloat16)
    gamma = torch.ones(512)
    x = wide.to(DEV)[:, 512:1024]                                  # row stride 1536
    got = add_rms_norm(x, gamma.to(DEV), 1e-5)
    _close(got, oracle.add_rms_norm_oracle(wide[:, 512:1024], gamma, 1e-5), torch.bfloat16)
    with pytest.raises(ValueError):
        add_rms_norm(x, gamma.to(DEV)[:100], 1e-5)
    with pytest.raises(ValueError):
        add_rms_norm(torch.zeros(2, 12, device=DEV), torch.ones(12, device=DEV), 1e-5)      # hidden % 8
    assert add_rms_norm(torch.zeros(0, 64, device=DEV), torch.ones(64, device=DEV), 1e-5).shape == (0, 64)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,width", [(64, 3072), (1, 8), (33, 1000), (1000, 512)])
def test_silu_and_mul(dtype, rows, width):
    g = torch.Generator().manual_seed(rows + width)
    x = (torch.randn(rows, 2 * width, generator=g) * 3).to(dtype)
    want = oracle.silu_and_mul_oracle(x)
    got = silu_and_mul(x.to(DEV))
    _close(got, want, dtype, ulps=2.0)      # one ulp of the rounded silu moves the product by up to one more
    # strided input rows (a slice of a wider buffer)
    wide = torch.zeros(rows, 2 * width + 64, dtype=dtype)
    wide[:, : 2 * width] = x
    _close(silu_and_mul(wide.to(DEV)[:, : 2 * width]), want, dtype, ulps=2.0)


def test_operators_run_on_the_current_stream():
    """What the operators take for the current stream is torch's: default, inside a stream's block, on another thread, under capture."""
    from concurrent.futures import ThreadPoolExecutor
    from minivllm_amd import _C
    device = torch.zeros(1, device=DEV).device
    same = lambda: _C.current_stream_ptr(device) == torch.cuda.current_stream(device).cuda_stream
    side = torch.cuda.Stream()
    assert same() and _C.current_stream_ptr(torch.device("cuda")) == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side), ThreadPoolExecutor(1) as pool:
        assert same() and _C.current_stream_ptr(device) == side.cuda_stream
        assert pool.submit(same).result() and pool.submit(_C.current_stream_ptr, device).result() != side.cuda_stream
    x, graph = torch.randn(4, 64, device=DEV), torch.cuda.CUDAGraph()
    gamma = torch.ones(64, device=DEV)
    add_rms_norm(x, gamma, 1e-6)
    with torch.cuda.graph(graph):
        assert same()
        y = add_rms_norm(x, gamma, 1e-6)
    x.copy_(torch.randn(4, 64, device=DEV))
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, add_rms_norm(x, gamma, 1e-6))
