"""S4ConvD, the model that calls the depthwise Conv1D path, with the block's
skip term fused into the convolution.

Follows the reference's S4 model (``kernels/warp_tiled_ampere.py:1116-1224``):
``S4ConvKernel`` builds the H x L convolution kernel from a diagonal
state-space parameterisation (:1122-1169), ``S4ConvBlock`` applies it with a
per-channel skip term, a GELU, dropout and a GLU output projection
(:1172-1190), ``Model`` stacks the blocks between a linear encoder and
decoder (:1193-1215), and ``rmsle`` is the training loss (:1218-1224).
Parameter names, shapes, registration order and initial distributions are
the reference's, so its checkpoints load unchanged.

The fused skip term. The block computes ``y = conv(x, k) + x * skip[h]``
(:1187-1188). The skip term reads ``x[b,h,t]``, which is what tap
``p = K // 2`` of the convolution reads (``y[t]`` gets ``w[p] * x[t+p-p]``).
So ``conv(x, k) + skip * x = conv(x, k')`` with ``k' = k`` plus ``skip`` on
column p, and the HIP path runs the block's FWD and dX with ``k'``: the skip
term costs no pass over ``y``. In backward, ``dL/dk = dK`` (``k' - k`` does
not depend on k) and ``dL/dskip = dK[:, p]``.

Backend switch: ``pathtile_amd.kernels.warp_tiled_ampere.TRAIN_CONV_BACKEND``
(the reference's module global, :1119), read on every forward call:
``"warp"`` runs the HIP path with the fused skip term, ``"pytorch"`` runs the
reference's composition (``reference_depthwise_conv`` + a separate skip add).
"""

from __future__ import annotations

import ctypes
import math
from typing import Any

import torch
from torch import nn

from . import _lib
from .runtime import (
    KERNEL_EVENTS, MAX_L, HipWarpRuntime, _call, _ptr, get_runtime, reference_depthwise_conv,
)


def _backend() -> str:
    from .kernels import warp_tiled_ampere

    return warp_tiled_ampere.TRAIN_CONV_BACKEND


class DepthConvSkipAmpere(torch.autograd.Function):
    """``conv(x, k) + x * skip[:, None]`` on the HIP path, the skip term
    folded into tap ``K // 2``; backward returns ``(gx, gk, gskip)`` with
    the two-pass deterministic dK."""

    @staticmethod
    def forward(ctx: Any, x: torch.Tensor, k: torch.Tensor, skip: torch.Tensor) -> torch.Tensor:
        runtime = get_runtime()
        x_c = x.contiguous()
        k_c = k.contiguous()
        B, H, L, K = runtime._check_shapes(x_c, k_c)
        if tuple(skip.shape) != (H,):
            raise ValueError(f"skip must have shape {(H,)}")
        if skip.dtype != torch.float32 or skip.device != k_c.device:
            raise ValueError("skip must be a float32 tensor on the kernel's device")
        p = K // 2
        k_eff = k_c.clone()
        k_eff[:, p] += skip
        y = torch.empty_like(x_c)
        runtime.launch_fwd(x_c, k_eff, y)
        ctx.save_for_backward(x_c, k_eff)
        ctx.params = (B, H, L, K)
        return y

    @staticmethod
    def backward(ctx: Any, gy: torch.Tensor):
        runtime = get_runtime()
        x_c, k_eff = ctx.saved_tensors
        B, H, L, K = ctx.params
        gy_c = gy.contiguous()
        gx = gk = gskip = None
        if (type(runtime) is HipWarpRuntime and ctx.needs_input_grad[0]
                and (ctx.needs_input_grad[1] or ctx.needs_input_grad[2])):
            gx, dk = torch.empty_like(x_c), torch.empty_like(k_eff)
            runtime.launch_backward(gy_c, x_c, k_eff, gx, dk)
            return (gx, dk if ctx.needs_input_grad[1] else None,
                    dk[:, K // 2].contiguous() if ctx.needs_input_grad[2] else None)
        if ctx.needs_input_grad[0]:
            gx = torch.empty_like(x_c)
            runtime.launch_bwd_input(gy_c, k_eff, gx)
        if ctx.needs_input_grad[1] or ctx.needs_input_grad[2]:
            dk = torch.empty_like(k_eff)
            runtime.launch_bwd_weight_deterministic(gy_c, x_c, dk, K)
            if ctx.needs_input_grad[1]:
                gk = dk
            if ctx.needs_input_grad[2]:
                gskip = dk[:, K // 2].contiguous()
        return gx, gk, gskip


def depthwise_conv_skip_ampere(x: torch.Tensor, k: torch.Tensor, skip: torch.Tensor) -> torch.Tensor:
    return DepthConvSkipAmpere.apply(x, k, skip)


def _taps(log_dt, C_re, C_im, log_A_re, A_im, taps: int,
          device: torch.device | None = None) -> torch.Tensor:
    dt = log_dt.exp()
    A = torch.complex(-log_A_re.exp(), A_im)
    C = torch.complex(C_re, C_im)
    dtA = A * dt[:, None]
    C_eff = C * (dtA.exp() - 1.0) / A
    t = torch.arange(taps, device=log_dt.device if device is None else device,
                     dtype=torch.float32)
    powers = torch.exp(dtA[:, :, None] * t)  # [H, N/2, taps]
    # elementwise product and sum over n (no batched matmul)
    return (2.0 * (C_eff[:, :, None] * powers).sum(dim=1).real).contiguous()


class S4ConvKernel(nn.Module):
    """Diagonal SSM convolution kernel (:1122-1169). For channel h and tap t:
    ``k[h, t] = 2 Re( sum_n C_eff[h, n] * exp(dt[h] A[h, n] t) )`` with
    ``A = -exp(log_A_re) + i A_im``, ``C = C_re + i C_im`` and
    ``C_eff = C (exp(dt A) - 1) / A`` (zero-order-hold discretisation)."""

    def __init__(self, hidden_dim: int, state_dim: int) -> None:
        super().__init__()
        self.H = hidden_dim
        self.N = state_dim
        half = state_dim // 2
        lo, hi = math.log(0.001), math.log(0.1)
        self.log_dt = nn.Parameter(torch.rand(hidden_dim) * (hi - lo) + lo)
        self.C_re = nn.Parameter(torch.randn(hidden_dim, half))
        self.C_im = nn.Parameter(torch.randn(hidden_dim, half))
        self.log_A_re = nn.Parameter(torch.randn(hidden_dim, half))
        self.A_im = nn.Parameter(torch.ones(hidden_dim, half))

    def build_kernel(self, taps: int, device: torch.device) -> torch.Tensor:
        return _taps(self.log_dt, self.C_re, self.C_im, self.log_A_re, self.A_im, taps, device)

    def forward(self, x: torch.Tensor, skip: torch.Tensor | None = None) -> torch.Tensor:
        """``conv(x, k)`` with ``k = build_kernel(L)``; with ``skip`` the block's
        skip term is added (fused into the convolution on the "warp" backend)."""
        _, H, L = x.shape
        if H != self.H:
            raise ValueError(f"Expected H={self.H}, got {H}")
        if L > MAX_L:
            raise ValueError(f"Warp-tiled paper kernel supports L<={MAX_L}")
        k = self.build_kernel(L, x.device)
        backend = _backend()
        if backend == "warp":
            if skip is None:
                from .runtime import depthwise_conv_ampere

                return depthwise_conv_ampere(x.contiguous(), k)
            return depthwise_conv_skip_ampere(x.contiguous(), k, skip)
        if backend == "pytorch":
            y = reference_depthwise_conv(x.contiguous(), k)
            return y if skip is None else y + x * skip.unsqueeze(-1)
        raise RuntimeError(f"Unknown training backend: {backend}")


# ---------------------------------------------------------------------------
# The whole block in fused HIP passes (pt_s4_block_*)
# ---------------------------------------------------------------------------
FUSED_MAX_H = 256  # H a multiple of 32 up to here
# The model's ends: channels (a multiple of 4), input features, outputs
ENDS_MAX_H, ENCODER_MAX_IN, HEAD_MAX_OUT = 1024, 8, 4


def _size_query(fn: str, *args: int) -> int:
    out = ctypes.c_size_t(0)
    _lib.check(getattr(_lib.load(), fn)(*args, ctypes.byref(out)), fn)
    return int(out.value)


def _dropout_mask(x: torch.Tensor, p: float) -> torch.Tensor | None:
    """The mask that the dropout module draws for the convolution's output in
    its [B, H, L] shape: PyTorch's own draw for a tensor of that shape, whose
    values (here the input's) it does not depend on."""
    if p == 0.0:
        return None
    B, L, H = x.shape
    return torch.native_dropout(x.detach().view(B, H, L), p, True)[1]


def _fused_mix(x: torch.Tensor, skip, log_dt, c_re, c_im, log_a_re, a_im, weight, mask,
               scale: float, backward: bool, x_copy: torch.Tensor | None = None):
    """Taps and split projection (prep) and the convolution's output after
    dropout, v [B, L, H]; x into x_copy."""
    runtime = get_runtime()
    runtime._check_open()
    B, L, H = x.shape
    prep = x.new_empty(_size_query("pt_s4_block_prep_values", H, L, c_re.shape[1]))
    v = torch.empty_like(x)
    _call(runtime._lib.pt_s4_block_mix_f32, x.device,
          _ptr(x), _ptr(log_dt), _ptr(c_re), _ptr(c_im), _ptr(log_a_re), _ptr(a_im),
          _ptr(skip), _ptr(weight), None if mask is None else _ptr(mask), scale, _ptr(prep),
          _ptr(v), None if x_copy is None else _ptr(x_copy), B, H, L, c_re.shape[1],
          int(backward))
    return prep, v


def _fused_tail(v: torch.Tensor, x: torch.Tensor, prep, weight, bias,
                q: torch.Tensor | None = None) -> torch.Tensor:
    runtime = get_runtime()
    B, L, H = x.shape
    y = torch.empty_like(x)
    _call(runtime._lib.pt_s4_block_tail_f32, x.device,
          _ptr(v), _ptr(x), _ptr(prep), _ptr(weight), _ptr(bias), _ptr(y),
          None if q is None else _ptr(q), B, H, L)
    return y


class S4BlockFused(torch.autograd.Function):
    """``S4ConvBlock.forward`` as one function of the input and the block's
    parameters: taps, convolution with the skip term, dropout, GELU,
    projection, GLU and residual, all in [B, L, H]. The backward reads x. With
    ``copy`` it reads a copy that the convolution writes on its way, so that
    x may change in between (``x += block(x)``; the separate operations save
    the copy that their transpose makes). The copy is a second output: that
    ties it to x for a backward that is differentiated. Of the parameters it
    saves those that the separate operations save as they are, so that the
    others may change as well: their values are in prep, and only a backward
    as torch's operations reads them again."""

    @staticmethod
    def forward(ctx: Any, x, skip, log_dt, c_re, c_im, log_a_re, a_im, weight, bias, p: float,
                copy: bool = False):
        mask = _dropout_mask(x, p)
        ctx.scale = 1.0 / (1.0 - p)
        ctx.set_materialize_grads(False)
        x_copy = torch.empty_like(x) if copy else None
        prep, v = _fused_mix(x, skip, log_dt, c_re, c_im, log_a_re, a_im, weight, mask,
                             ctx.scale, True, x_copy)
        q = x.new_empty((2, *x.shape))
        y = _fused_tail(v, x, prep, weight, bias, q)
        saved = (x_copy if copy else x, c_re, c_im, a_im, weight, prep, v, q, mask)
        ctx.forms = [_form(t) for t in saved]
        ctx.save_for_backward(*saved)
        ctx.unsaved = skip, log_dt, log_a_re, bias
        ctx.versions = _versions(ctx.unsaved)
        return (y, x_copy) if copy else y

    @staticmethod
    def backward(ctx: Any, gy: torch.Tensor | None, g_copy: torch.Tensor | None = None):
        grads = [None] * len(ctx.needs_input_grad)
        if gy is not None:
            grads[:9] = S4BlockFused._backward(ctx, gy)
        if g_copy is not None and ctx.needs_input_grad[0]:
            grads[0] = g_copy if grads[0] is None else grads[0] + g_copy
        return tuple(grads)

    @staticmethod
    def _backward(ctx: Any, gy: torch.Tensor):
        saved = ctx.saved_tensors
        need = ctx.needs_input_grad[:9]
        if _as_operations(gy):
            return _composed_grads(ctx, gy)
        x, c_re, c_im, a_im, weight, prep, v, q, mask = map(_unpacked, saved, ctx.forms)
        skip, log_dt, log_a_re, bias = ctx.unsaved
        runtime = get_runtime()
        runtime._check_open()
        B, L, H = x.shape
        gy = _aligned(gy.contiguous())
        gx = torch.empty_like(x) if need[0] else None
        taps = any(need[1:7])
        gp = [torch.empty_like(t) for t in (log_dt, c_re, c_im, log_a_re, a_im, skip)] \
            if taps else [None] * 6
        proj = need[7] or need[8]
        gw, gb = (torch.empty_like(weight), torch.empty_like(bias)) if proj else (None, None)
        nbytes = _size_query("pt_s4_block_bwd_workspace_bytes", B, H, L)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)

        def opt(t):
            return None if t is None else _ptr(t)

        _call(runtime._lib.pt_s4_block_bwd_f32, x.device,
              _ptr(gy), _ptr(x), _ptr(v), _ptr(q), opt(mask), ctx.scale, _ptr(prep),
              _ptr(weight), _ptr(c_re), _ptr(c_im), _ptr(a_im), opt(gx), *(opt(t) for t in gp),
              opt(gw), opt(gb), _ptr(ws), nbytes, B, H, L, c_re.shape[1])
        grads = [gx, gp[5], *gp[:5], gw, gb]
        return [g if n else None for g, n in zip(grads, need)]


def _versions(tensors) -> list:
    return [None if t.is_inference() else t._version for t in tensors]


def _as_operations(gy: torch.Tensor) -> bool:
    """The backward runs as torch's operations instead of the kernels: it is
    itself differentiated (create_graph), or `gy` is a batch of gradients
    (is_grads_batched, vmap over the backward), which has no address."""
    return (torch.is_grad_enabled() or torch._C._functorch.is_legacy_batchedtensor(gy)
            or torch._C._functorch.is_functorch_wrapped_tensor(gy))


def _composed_grads(ctx: Any, gy: torch.Tensor):
    """The block's gradients through torch's operations on the saved inputs
    (the convolution's own backward stays first order and takes one gradient,
    as its autograd function is). They are taken at aliases: where x was
    computed from the same parameters, as in a block applied twice, a gradient
    with respect to the tensors themselves would follow that path too, which
    the engine adds by itself."""
    create_graph = torch.is_grad_enabled()
    need = ctx.needs_input_grad[:9]
    x, c_re, c_im, a_im, weight, _, v, _, mask = ctx.saved_tensors
    skip, log_dt, log_a_re, bias = ctx.unsaved
    if _versions(ctx.unsaved) != ctx.versions:
        raise RuntimeError("a parameter of the block was modified by an inplace operation "
                           "before a backward that is differentiated")
    with torch.enable_grad():
        inputs = [t.view_as(t) if n else t.detach() for t, n in zip(
            (x, skip, log_dt, c_re, c_im, log_a_re, a_im, weight, bias), need)]
        x, skip, log_dt, c_re, c_im, log_a_re, a_im, weight, bias = inputs
        if any(need[:7]):
            k = _taps(log_dt, c_re, c_im, log_a_re, a_im, x.shape[1])
            v = depthwise_conv_skip_ampere(x.transpose(1, 2).contiguous(), k, skip)
            if mask is not None:
                v = v * mask * ctx.scale
        else:  # the forward's, without a convolution that vmap cannot enter
            v = v.detach().transpose(1, 2)
        z = nn.functional.conv1d(nn.functional.gelu(v), weight, bias)
        y = nn.functional.glu(z, dim=1).transpose(1, 2) + x
        got = iter(torch.autograd.grad(y, [t for t, n in zip(inputs, need) if n], gy,
                                       create_graph=create_graph))
    return [next(got) if n else None for n in need]


def _free_choice(runtime: Any) -> bool:
    """Nobody has a say in the convolution's launches: the runtime is the
    framework's own class (another may replace any launch) and neither it nor
    the environment names a kernel."""
    return (type(runtime) is HipWarpRuntime and runtime.rows_algo == "auto"
            and not runtime._lib.pt_kernel_choice_forced())


def _no_hooks(m: nn.Module) -> bool:
    return not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks
                or m._backward_pre_hooks or "forward" in m.__dict__)


def _tracing() -> bool:
    """True where something watches or rewrites the block's single operations:
    compilers and tracers, functorch transforms, forward-mode AD, dispatch and
    function modes (but the default-device one), autocast, module hooks."""
    if torch.compiler.is_compiling():  # first: a compiler cannot trace the rest
        return True
    if torch._C._len_torch_function_stack():
        from torch.overrides import _get_current_function_mode_stack
        from torch.utils._device import DeviceContext

        if any(type(m) is not DeviceContext for m in _get_current_function_mode_stack()):
            return True
    return bool(torch._C._len_torch_dispatch_stack()
                or torch.autograd.forward_ad._current_level >= 0
                or torch._C._functorch.peek_interpreter_stack() is not None
                or torch.is_autocast_enabled("cuda")
                or torch.jit.is_tracing()
                or nn.modules.module._has_any_global_hook())


class EncoderFused(torch.autograd.Function):
    """``nn.Linear`` over up to 8 input features: one pass over the output, and
    one over its gradient for the weight and bias gradients. Like the module
    it saves x for the weight's gradient and the weight for x's, and neither
    where nobody asks."""

    @staticmethod
    def forward(ctx: Any, x, weight, bias):
        B, L, n = x.shape
        H = weight.shape[0]
        y = x.new_empty((B, L, H))
        _call(_lib.load().pt_s4_encode_f32, x.device,
              _ptr(x), _ptr(weight), _ptr(bias), _ptr(y), B, L, n, H)
        need = ctx.needs_input_grad
        saved = (x if need[1] else None, weight if need[0] else None)
        ctx.forms = [_form(t) for t in saved]
        ctx.save_for_backward(*saved)
        return y

    @staticmethod
    def backward(ctx: Any, gy: torch.Tensor):
        x, weight = ctx.saved_tensors
        need = ctx.needs_input_grad
        gx = gy @ weight if need[0] else None
        if not need[1] or _as_operations(gy):
            return (gx, (gy.unsqueeze(-1) * x.unsqueeze(-2)).sum((0, 1)) if need[1] else None,
                    gy.sum((0, 1)) if need[2] else None)
        x = _unpacked(x, ctx.forms[0])
        B, L, n = x.shape
        H = gy.shape[2]
        gy = _aligned(gy.contiguous())
        gw, gb = gy.new_empty((H, n)), gy.new_empty(H)
        nbytes = _size_query("pt_s4_encode_grad_workspace_bytes", B, L, n, H)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
        _call(_lib.load().pt_s4_encode_grad_f32, x.device,
              _ptr(x), _ptr(gy), _ptr(gw), _ptr(gb), _ptr(ws), nbytes, B, L, n, H)
        return gx, gw, gb if need[2] else None


class HeadFused(torch.autograd.Function):
    """The decoder at the last column, ``decoder(x)[:, -1, :]``: the columns
    before it reach neither the output nor a gradient. Saves what the module
    does (EncoderFused)."""

    @staticmethod
    def forward(ctx: Any, x, weight, bias):
        B, L, H = x.shape
        n = weight.shape[0]
        out = x.new_empty((B, n))
        _call(_lib.load().pt_s4_head_f32, x.device,
              _ptr(x), _ptr(weight), _ptr(bias), _ptr(out), B, H, L, n)
        need = ctx.needs_input_grad
        saved = (x if need[1] else None, weight if need[0] else None)
        ctx.shape = x.shape
        ctx.forms = [_form(t) for t in saved]
        ctx.save_for_backward(*saved)
        return out

    @staticmethod
    def backward(ctx: Any, gy: torch.Tensor):
        x, weight = ctx.saved_tensors
        need = ctx.needs_input_grad
        B, L, H = ctx.shape
        if not need[1] or _as_operations(gy):
            gx = nn.functional.pad((gy @ weight)[:, None, :], (0, 0, L - 1, 0)) if need[0] else None
            return (gx, gy.t() @ x[:, -1, :] if need[1] else None,
                    gy.sum(0) if need[2] else None)
        x, weight = map(_unpacked, (x, weight), ctx.forms)
        n = gy.shape[1]
        gy = gy.contiguous()
        gx = torch.empty_like(x) if need[0] else None
        gw, gb = gy.new_empty((n, H)), gy.new_empty(n)
        nbytes = _size_query("pt_s4_head_grad_workspace_bytes", B, H, L, n)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
        _call(_lib.load().pt_s4_head_grad_f32, x.device,
              _ptr(x), _ptr(gy), None if weight is None else _ptr(weight),
              None if gx is None else _ptr(gx), _ptr(gw), _ptr(gb), _ptr(ws), nbytes, B, H, L, n)
        return gx, gw, gb if need[2] else None


def _aligned(t: torch.Tensor) -> torch.Tensor:
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _form(t: torch.Tensor | None):
    return None if t is None else (t.shape, t.dtype, t.device)


def _unpacked(t: torch.Tensor | None, form):
    """A saved tensor for a kernel that takes its address: a saved-tensor hook
    may give back other strides or another alignment (copied), or another
    shape, type or device than the `_form` it was saved in (refused)."""
    if _form(t) != form:
        raise RuntimeError(f"saved tensor {form} was unpacked as {_form(t)}")
    return None if t is None else _aligned(t.contiguous())


def _whole_linear(m: nn.Module) -> bool:
    """`m` is an ordinary FP32 ``nn.Linear`` whose call nothing watches, with
    one bias value per row of its weight, as the kernels read them
    (``F.linear`` broadcasts fewer). The sizes are the tensors' own:
    ``out_features`` does not follow a replaced weight."""
    if not (type(m) is nn.Linear and _no_hooks(m)):
        return False
    w, b = m.weight, m.bias
    return (b is not None and w.dim() == 2 and b.shape == w.shape[:1]
            and all(type(t) in (nn.Parameter, torch.Tensor) and t.dtype == torch.float32
                    and t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (w, b)))


def _plain_linear(m: nn.Module, x: torch.Tensor) -> bool:
    """`m` is a `_whole_linear` for the contiguous GPU tensor `x` [B, L, width]."""
    if not (type(x) is torch.Tensor and x.is_cuda and x.dim() == 3
            and x.dtype == torch.float32 and x.is_contiguous() and x.data_ptr() % 16 == 0
            and 0 < x.numel() < 2**31 and _backend() == "warp" and _whole_linear(m)):
        return False
    w = m.weight
    return x.shape[2] == w.shape[1] and w.device == x.device and m.bias.device == x.device


def _end_served(x: torch.Tensor, channels: int) -> bool:
    """The ends' kernels serve `channels` channels at the columns of `x`."""
    return (4 <= channels <= ENDS_MAX_H and channels % 4 == 0
            and x.shape[0] * x.shape[1] * channels < 2**31)


class S4ConvBlock(nn.Module):
    """Depthwise S4 convolution + skip, GELU, dropout, GLU projection and a
    residual connection (:1172-1190); input and output are ``[B, L, H]``."""

    def __init__(self, hidden_dim: int, state_dim: int, dropout: float) -> None:
        super().__init__()
        self.skip = nn.Parameter(torch.randn(hidden_dim))
        self.kernel_layer = S4ConvKernel(hidden_dim, state_dim)
        self.activation = nn.GELU()
        self.dropout = nn.Dropout(dropout)
        self.output_linear = nn.Sequential(
            nn.Conv1d(hidden_dim, 2 * hidden_dim, kernel_size=1),
            nn.GLU(dim=1),
        )

    def _fused_inputs(self, x: torch.Tensor):
        """The parameters in S4BlockFused's order, or None where the block
        runs as separate operations: another backend, layout, type or device,
        a shape the fused passes do not serve, modules that were replaced,
        subclassed or hooked, kernel timing through KERNEL_EVENTS (its phases
        are the separate launches), a runtime of the caller's own or a kernel
        choice (`_free_choice`), or tracing of any kind."""
        if _tracing():  # before the rest, which a tracer cannot follow
            return None
        kl, act, drop, out = self.kernel_layer, self.activation, self.dropout, self.output_linear
        if not (type(x) is torch.Tensor and x.dim() == 3 and x.is_cuda
                and type(kl) is S4ConvKernel and type(act) is nn.GELU
                and "build_kernel" not in kl.__dict__ and act.approximate == "none"
                and type(drop) is nn.Dropout and not drop.inplace and 0.0 <= drop.p < 1.0
                and type(out) is nn.Sequential and len(out) == 2):
            return None
        conv, glu = out  # a module's attribute costs half a microsecond: each once
        if not (type(conv) is nn.Conv1d and type(glu) is nn.GLU and glu.dim == 1):
            return None
        B, L, H = x.shape
        params = (self.skip, kl.log_dt, kl.C_re, kl.C_im, kl.log_A_re, kl.A_im, conv.weight,
                  conv.bias)
        half, bias = params[2].shape[-1] if params[2].dim() == 2 else 0, params[7]
        shapes = ((H,), (H,), (H, half), (H, half), (H, half), (H, half), (2 * H, H, 1), (2 * H,))
        if not (x.dtype == torch.float32 and x.is_contiguous() and x.data_ptr() % 16 == 0
                and 1 <= L <= MAX_L and 32 <= H <= FUSED_MAX_H and H % 32 == 0 and kl.H == H
                and half >= 1 and B >= 1 and x.numel() < 2**31
                and conv.groups == 1 and conv.stride == (1,) and conv.padding == (0,)
                and bias is not None and _backend() == "warp"
                and not KERNEL_EVENTS.enabled and _free_choice(get_runtime())):
            return None
        for t, shape in zip(params, shapes):
            if not (type(t) in (nn.Parameter, torch.Tensor) and t.dtype == torch.float32
                    and t.device == x.device and t.shape == shape and t.is_contiguous()):
                return None
        if bias.data_ptr() % 16:
            return None
        if not all(_no_hooks(m) for m in (kl, act, drop, out, conv, glu)):
            return None
        return params

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        params = self._fused_inputs(x)
        if params is not None:
            p = float(self.dropout.p) if self.dropout.training else 0.0
            if torch.is_grad_enabled() and (x.requires_grad
                                            or any(t.requires_grad for t in params)):
                if getattr(x, "_held_by_model_alone", False):
                    return S4BlockFused.apply(x, *params, p)
                return S4BlockFused.apply(x, *params, p, True)[0]
            skip, *kernel, weight, bias = params
            mask = _dropout_mask(x, p)
            prep, v = _fused_mix(x, skip, *kernel, weight, mask, 1.0 / (1.0 - p), False)
            return _fused_tail(v, x, prep, weight, bias)
        x_hl = x.transpose(1, 2).contiguous()
        y = self.kernel_layer(x_hl, self.skip)
        y = self.output_linear(self.activation(self.dropout(y)))
        return y.transpose(1, 2) + x


class Model(nn.Module):
    """Encoder, ``num_blocks`` S4ConvD blocks, decoder; ``x`` is
    ``[B, L, input_dim]`` and the output is the last step's ``[B, output_dim]``
    (:1193-1215)."""

    def __init__(
        self,
        state_dim: int = 64,
        hidden_dim: int = 128,
        input_dim: int = 4,
        output_dim: int = 1,
        num_blocks: int = 4,
        dropout: float = 0.01,
    ) -> None:
        super().__init__()
        self.encoder = nn.Linear(input_dim, hidden_dim)
        self.blocks = nn.ModuleList(
            [S4ConvBlock(hidden_dim, state_dim, dropout) for _ in range(num_blocks)]
        )
        self.decoder = nn.Linear(hidden_dim, output_dim)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        plain = not _tracing()
        saving = plain and torch.is_grad_enabled()
        enc, dec = self.encoder, self.decoder
        if plain and _plain_linear(enc, x) and x.shape[2] <= ENCODER_MAX_IN and _end_served(
                x, enc.weight.shape[0]):
            x = EncoderFused.apply(x, enc.weight, enc.bias)
            held = saving  # x is a new tensor that nothing else has seen
        else:
            x = enc(x)
            held = saving and type(enc) is nn.Linear and _no_hooks(enc)
        for block in self.blocks:
            unseen = saving and type(block) is S4ConvBlock and _no_hooks(block)
            if held and unseen:
                x._held_by_model_alone = True
            x = block(x)
            held = unseen
        if plain and _plain_linear(dec, x) and dec.weight.shape[0] <= HEAD_MAX_OUT and _end_served(
                x, x.shape[2]):
            return HeadFused.apply(x, dec.weight, dec.bias)
        return dec(x)[:, -1, :]


def rmsle(prediction: torch.Tensor, target: torch.Tensor) -> torch.Tensor:
    """Root mean squared log error on non-negative parts (:1218-1224)."""
    p = prediction.reshape(-1).clamp(min=0.0)
    t = target.reshape(-1).clamp(min=0.0)
    return torch.sqrt((p.log1p() - t.log1p()).square().mean() + 1e-12)


__all__ = [
    "DepthConvSkipAmpere", "depthwise_conv_skip_ampere",
    "S4ConvKernel", "S4ConvBlock", "Model", "rmsle",
]
