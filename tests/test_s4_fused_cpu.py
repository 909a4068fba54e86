"""The host side of the S4ConvD block's fused functions, without a GPU: what
they allocate, differentiate and hand to the kernels, with the native calls
replaced (kernels/warp_tiled_ampere.py:1122-1215 is the module that they
serve). The kernels themselves are in test_gpu_s4_block.py."""

from __future__ import annotations

import pytest
import torch

from pathtile_amd import runtime, s4convd


@pytest.fixture
def calls(monkeypatch):
    """Installs a runtime and records the native calls instead of making
    them; yields the list of (function name, arguments)."""
    seen = []
    monkeypatch.setattr(runtime, "_RUNTIME", runtime.HipWarpRuntime())
    monkeypatch.setattr(s4convd, "_call",
                        lambda fn, device, *args: seen.append((fn.__name__, args)))
    return seen


@pytest.fixture
def default_dtype():
    old = torch.get_default_dtype()
    yield torch.set_default_dtype
    torch.set_default_dtype(old)


def _f32(*shape):
    return torch.randn(*shape, dtype=torch.float32)


def _block_inputs(B, L, H, half):
    return (_f32(B, L, H), _f32(H), _f32(H), *(_f32(H, half) for _ in range(4)),
            _f32(2 * H, H, 1), _f32(2 * H))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float64])
def test_buffers_are_fp32_under_any_default_dtype(calls, default_dtype, dtype):
    """The kernels write FP32 into every buffer, whatever type torch gives to
    tensors that name none: outputs, saved values and gradients."""
    default_dtype(dtype)
    B, L, H, half = 3, 5, 32, 4
    inputs = tuple(t.requires_grad_(True) for t in _block_inputs(B, L, H, half))
    y = s4convd.S4BlockFused.apply(*inputs, 0.0)
    prep, v, q = y.grad_fn.saved_tensors[9:12]
    for t in (y, prep, v, q, *torch.autograd.grad(y, inputs, torch.ones_like(y))):
        assert t.dtype == torch.float32
    assert q.shape == (2, B, L, H)
    x, w, b = (t.requires_grad_(True) for t in (_f32(B, L, 4), _f32(H, 4), _f32(H)))
    y = s4convd.EncoderFused.apply(x, w, b)
    for t in (y, *torch.autograd.grad(y, (w, b), torch.ones_like(y))):
        assert t.dtype == torch.float32
    h, w, b = (t.requires_grad_(True) for t in (_f32(B, L, H), _f32(2, H), _f32(2)))
    out = s4convd.HeadFused.apply(h, w, b)
    for t in (out, *torch.autograd.grad(out, (h, w, b), torch.ones_like(out))):
        assert t.dtype == torch.float32
    assert {n for n, _ in calls} == {
        "pt_s4_block_mix_f32", "pt_s4_block_tail_f32", "pt_s4_block_bwd_f32", "pt_s4_encode_f32",
        "pt_s4_encode_grad_f32", "pt_s4_head_f32", "pt_s4_head_grad_f32"}
