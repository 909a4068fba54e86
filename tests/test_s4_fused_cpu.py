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
    prep, v, q = y.grad_fn.saved_tensors[5:8]
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


@pytest.fixture
def composed(monkeypatch):
    """Native forward passes of the block replaced by the operations they
    fuse, and the convolution by a differentiable one."""
    def conv(x, k, skip):
        return s4convd.reference_depthwise_conv(x, k) + x * skip.unsqueeze(-1)

    def mix(x, skip, log_dt, c_re, c_im, log_a_re, a_im, weight, mask, scale, backward,
            x_copy=None):
        if x_copy is not None:
            x_copy.copy_(x)
        k = s4convd._taps(log_dt, c_re, c_im, log_a_re, a_im, x.shape[1])
        v = conv(x.transpose(1, 2), k, skip)
        if mask is not None:
            v = v * mask * scale
        return x.new_empty(0), v.transpose(1, 2).contiguous()

    def tail(v, x, prep, weight, bias, q=None):
        z = torch.nn.functional.conv1d(torch.nn.functional.gelu(v.transpose(1, 2)), weight, bias)
        return torch.nn.functional.glu(z, dim=1).transpose(1, 2) + x

    monkeypatch.setattr(s4convd, "depthwise_conv_skip_ampere", conv)
    monkeypatch.setattr(s4convd, "_fused_mix", mix)
    monkeypatch.setattr(s4convd, "_fused_tail", tail)


@pytest.mark.parametrize("copy", [False, True])
@pytest.mark.parametrize("applications", [1, 2, 3])
def test_weight_tied_blocks_keep_their_gradients_under_create_graph(calls, composed, applications,
                                                                    copy):
    """One block applied several times: gradients with create_graph equal
    those of the separate operations (FP64), and so do second derivatives."""
    torch.manual_seed(applications)
    B, L, H, half = 3, 7, 32, 4
    inputs = [t.double().requires_grad_(True) for t in _block_inputs(B, L, H, half)]

    def grads(block):
        y = inputs[0]
        for _ in range(applications):
            y = block(y, *inputs[1:])
        gs = torch.autograd.grad(y.square().sum(), inputs, create_graph=True)
        # create_graph again, so that no native backward runs
        second = torch.autograd.grad(sum(g.square().sum() for g in gs), inputs, create_graph=True)
        return [g.detach() for g in (*gs, *second)]

    def separate(x, skip, log_dt, c_re, c_im, log_a_re, a_im, weight, bias):
        _, v = s4convd._fused_mix(x, skip, log_dt, c_re, c_im, log_a_re, a_im, weight, None, 1.0,
                                  True)
        return s4convd._fused_tail(v, x, None, weight, bias)

    def fused_block(*t):
        y = s4convd.S4BlockFused.apply(*t, 0.0, copy)
        return y[0] if copy else y

    for a, b in zip(grads(fused_block), grads(separate)):
        assert float((a - b).norm() / b.norm()) < 1e-10


def _linear(how):
    m = torch.nn.Linear(8, 12)
    if how == "one bias":  # F.linear broadcasts it
        m.bias = torch.nn.Parameter(torch.randn(1))
    elif how == "short bias":
        m.bias = torch.nn.Parameter(torch.randn(4))
    elif how == "vector":
        m.weight = torch.nn.Parameter(torch.randn(8))
    elif how == "no bias":
        m.bias = None
    elif how == "double":
        m.double()
    elif how == "transposed":
        m.weight = torch.nn.Parameter(torch.randn(8, 12).t())
    elif how == "misaligned":
        m.bias = torch.nn.Parameter(torch.randn(13)[1:])
    elif how == "hook":
        m.register_forward_hook(lambda *a: None)
    elif how == "replaced":  # whole, with other sizes than out_features says
        m.weight = torch.nn.Parameter(torch.randn(20, 8))
        m.bias = torch.nn.Parameter(torch.randn(20))
    return m


@pytest.mark.parametrize("how", ["one bias", "short bias", "vector", "no bias", "double",
                                 "transposed", "misaligned", "hook"])
def test_linear_modules_that_the_kernels_cannot_read(how):
    """Modules that run as themselves: their weight and bias are not what the
    ends' kernels read, one value per output among them."""
    assert not s4convd._whole_linear(_linear(how))


def test_linear_modules_are_taken_by_their_tensors():
    assert s4convd._whole_linear(_linear("as made"))
    assert s4convd._whole_linear(_linear("replaced"))
    x = torch.empty(3, 5, 4, device="meta")
    assert s4convd._end_served(x, 1024) and s4convd._end_served(x, 4)
    for channels in (0, 2, 6, 1028):
        assert not s4convd._end_served(x, channels)
    assert not s4convd._end_served(torch.empty(2**20, 2, 1, device="meta"), 1024)


@pytest.fixture
def pytorch_model(monkeypatch):
    from pathtile_amd.kernels import warp_tiled_ampere as wta

    monkeypatch.setattr(wta, "TRAIN_CONV_BACKEND", "pytorch")
    torch.manual_seed(2)
    return s4convd.Model(state_dim=8, hidden_dim=32, num_blocks=2, dropout=0.0)


@pytest.mark.parametrize("how", ["compile", "export", "fx", "jit", "vmap"])
def test_model_can_be_traced(pytorch_model, how):
    """The choice of the fused functions leaves the model to tracers: one
    whole graph for the compiler, and module graphs with the blocks as
    leaves."""
    m, x = pytorch_model.eval(), torch.randn(3, 20, 4)
    with torch.no_grad():
        ref = m(x)
        if how == "compile":
            torch._dynamo.reset()
            got = torch.compile(m, fullgraph=True, backend="eager")(x)
        elif how == "export":
            got = torch.export.export(m, (x,), strict=True).module()(x)
        elif how == "fx":
            class Blocks(torch.fx.Tracer):
                def is_leaf_module(self, mod, name):
                    return isinstance(mod, s4convd.S4ConvBlock) or super().is_leaf_module(mod, name)

            got = torch.fx.GraphModule(m, Blocks().trace(m))(x)
        elif how == "jit":
            got = torch.jit.trace(m, x)(x)
        else:
            got = torch.vmap(m)(x[None])[0]
    assert torch.allclose(got, ref, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("name,value", [("PATHTILE_ROWS_ALGO", "valu"),
                                        ("PATHTILE_ROWS_CHANNELS", "8"),
                                        ("PATHTILE_DK_ALGO", "valu")])
def test_a_kernel_choice_reaches_the_launches(monkeypatch, name, value):
    """A choice of the environment or of the runtime, and a runtime of the
    caller's own, rule the fused block out."""
    class Own(runtime.HipWarpRuntime):
        pass

    for n in ("PATHTILE_ROWS_ALGO", "PATHTILE_ROWS_CHANNELS", "PATHTILE_DK_ALGO"):
        monkeypatch.delenv(n, raising=False)
    rt = runtime.HipWarpRuntime()
    assert s4convd._free_choice(rt)
    assert not s4convd._free_choice(Own()) and not s4convd._free_choice(object())
    for algo in ("valu", "mfma"):
        assert not s4convd._free_choice(runtime.HipWarpRuntime(rows_algo=algo))
    monkeypatch.setenv(name, value)
    assert not s4convd._free_choice(rt)
    monkeypatch.delenv(name)
    assert s4convd._free_choice(rt)


@pytest.mark.parametrize("how", ["is_grads_batched", "vmap"])
def test_batches_of_gradients(calls, composed, how):
    """Each gradient of the batch by itself, for the block and the model's
    ends."""
    torch.manual_seed(11)
    B, L, H, n = 2, 6, 32, 3
    inputs = [t.double().requires_grad_(True) for t in _block_inputs(B, L, H, 4)]
    y = s4convd.S4BlockFused.apply(*inputs, 0.0)
    x, w, b = (t.double().requires_grad_(True) for t in (_f32(B, L, 4), _f32(H, 4), _f32(H)))
    e = s4convd.EncoderFused.apply(x, w, b)
    h, dw, db = (t.double().requires_grad_(True) for t in (_f32(B, L, H), _f32(2, H), _f32(2)))
    o = s4convd.HeadFused.apply(h, dw, db)
    for out, wrt in ((y, inputs), (e, (x, w, b)), (o, (h, dw, db))):
        gys = torch.randn(n, *out.shape, dtype=out.dtype)
        before = len(calls)
        if how == "vmap":
            batch = torch.vmap(lambda g: torch.autograd.grad(out, wrt, g, retain_graph=True))(gys)
        else:
            batch = torch.autograd.grad(out, wrt, gys, is_grads_batched=True, retain_graph=True)
        assert len(calls) == before  # no kernel saw the batch
        for i in range(n):
            ones = torch.autograd.grad(out, wrt, gys[i], create_graph=True)
            for a, g in zip(batch, ones):
                assert torch.allclose(a[i], g, rtol=1e-10, atol=1e-12)


@pytest.fixture
def fused(calls, composed, monkeypatch):
    """Blocks and ends take their fused functions on the CPU."""
    def params(block, x):
        kl, conv = block.kernel_layer, block.output_linear[0]
        return (block.skip, kl.log_dt, kl.C_re, kl.C_im, kl.log_A_re, kl.A_im, conv.weight,
                conv.bias)

    monkeypatch.setattr(s4convd.S4ConvBlock, "_fused_inputs", params)
    monkeypatch.setattr(s4convd, "_plain_linear", lambda m, x: s4convd._whole_linear(m))


def test_a_blocks_input_may_change_before_its_backward(fused):
    """``x += block(x)``: the block's gradients are those at the values that
    it saw."""
    torch.manual_seed(12)
    block = s4convd.S4ConvBlock(32, 8, 0.0)
    x = torch.randn(3, 6, 32)

    def grads(change):
        h = x.clone()
        y = block(h)
        if change:
            h += y.detach()
        return torch.autograd.grad(y.sum(), tuple(block.parameters()), create_graph=True)

    for a, b in zip(grads(True), grads(False)):
        assert torch.equal(a, b)


def _copies(out):
    seen, todo = set(), [out.grad_fn]
    while todo:
        f = todo.pop()
        if f is not None and f not in seen:
            seen.add(f)
            todo += [g for g, _ in f.next_functions]
    return sum(len(f.needs_input_grad) == 11 for f in seen if f.name() == "S4BlockFusedBackward")


@pytest.mark.parametrize("how,copies", [("plain", 0), ("encoder hook", 1), ("block hook", 2),
                                        ("identity encoder", 1)])
def test_the_models_own_activations_are_not_copied(fused, how, copies):
    """Between the modules of a model only it holds an activation, unless a
    module is hooked (its input and output are then seen) or replaced."""
    m = s4convd.Model(state_dim=8, hidden_dim=32, input_dim=8, num_blocks=3, dropout=0.0)
    if how == "encoder hook":
        m.encoder.register_forward_hook(lambda *a: None)
    elif how == "block hook":
        m.blocks[1].register_forward_hook(lambda *a: None)
    elif how == "identity encoder":
        m.encoder = torch.nn.Identity()
    x = torch.randn(2, 6, 32 if how == "identity encoder" else 8)
    x.requires_grad_(how == "identity encoder")
    assert _copies(m(x)) == copies


@pytest.mark.parametrize("end", ["EncoderFused", "HeadFused"])
def test_the_ends_save_what_their_gradients_read(calls, end):
    """As nn.Linear: x for the weight's gradient, the weight for x's. What no
    gradient reads may change before the backward."""
    fn, n = getattr(s4convd, end), 8 if end == "EncoderFused" else 2
    for needs in range(8):
        x, w, b = _f32(3, 5, 4), _f32(n, 4), _f32(n)
        for i, t in enumerate((x, w, b)):
            t.requires_grad_(bool(needs >> i & 1))
        out = fn.apply(x, w, b)
        if not needs:
            assert out.grad_fn is None
            continue
        with torch.no_grad():
            if not w.requires_grad:
                x += 1
            if not x.requires_grad:
                w += 1
            b += 1
        wrt = [t for t in (x, w, b) if t.requires_grad]
        for g, t in zip(torch.autograd.grad(out, wrt, torch.ones_like(out)), wrt):
            assert g.shape == t.shape and g.dtype == torch.float32


def test_gelu_polynomial_against_a_new_fit():
    """The coefficients in s4_kernels.hpp: their error in FP64, and that of a
    fit by the method that the comment there names (Lawson's iteration for
    the weighted minimax, one coefficient rounded at a time)."""
    import re
    from pathlib import Path

    import numpy as np
    from scipy.special import erfcx

    text = (Path(s4convd.__file__).parent / "csrc" / "s4_kernels.hpp").read_text()
    body = text[text.index("NormalCdf normal_cdf"):text.index("float gelu_f")]
    have = [float(c) for c in re.findall(r"(?:r = |t, )(-?[\d.]+)f[;)]", body)
            if abs(float(c)) < 1.0][::-1]
    assert len(have) == 8

    def parts(a):
        t = 1 / (1 + 9 / 32 * a)
        return t, np.maximum(1, a) * np.exp(-a * a / 2), erfcx(a / np.sqrt(2)) / 2

    def worst(c):
        t, w, r = parts(np.linspace(0, 20, 100001))
        return np.abs(w * (t * np.polynomial.polynomial.polyval(t, c) - r)).max()

    def fit(fixed):
        t, w, r = parts(np.linspace(0, 8, 2001))
        n = len(fixed)
        A = np.stack([w * t * t**k for k in range(n, 8)], 1)
        b = w * (r - t * np.polynomial.polynomial.polyval(t, fixed or [0.0]))
        p, best = np.ones(len(t)), (np.inf, None)
        for _ in range(300):
            c = np.linalg.lstsq(A * np.sqrt(p)[:, None], b * np.sqrt(p), rcond=None)[0]
            e = np.abs(A @ c - b)
            best = min(best, (e.max(), list(c)), key=lambda q: q[0])
            p = p * e / (p * e).sum()
        return best

    fixed = []
    for _ in range(8):
        fixed.append(float(np.float32(fit(fixed)[1][0])))
    assert fit([])[0] < 2.2e-10
    assert worst(have) < 4e-10 and worst(have) < 1.2 * worst(fixed)
    np.testing.assert_allclose(have, fixed, rtol=1e-4)


def test_projections_gradients_need_no_second_convolution(calls, composed, monkeypatch):
    """Batched gradients of the projection alone come from the forward's
    values: vmap cannot enter the convolution's autograd function."""
    torch.manual_seed(13)
    inputs = [t.double() for t in _block_inputs(2, 6, 32, 4)]
    wrt = [t.requires_grad_(True) for t in inputs[7:]]
    y = s4convd.S4BlockFused.apply(*inputs, 0.5)

    def refuse(*args):
        raise AssertionError("a convolution ran")

    monkeypatch.setattr(s4convd, "depthwise_conv_skip_ampere", refuse)
    gys = torch.randn(3, *y.shape, dtype=y.dtype)
    batch = torch.vmap(lambda g: torch.autograd.grad(y, wrt, g, retain_graph=True))(gys)
    for i in range(3):
        ones = torch.autograd.grad(y, wrt, gys[i], create_graph=True)
        for a, g in zip(batch, ones):
            assert torch.allclose(a[i], g, rtol=1e-10, atol=1e-12)


PARAMETERS = ("skip", "log_dt", "c_re", "c_im", "log_a_re", "a_im", "weight", "bias")


@pytest.mark.parametrize("create_graph", [False, True])
@pytest.mark.parametrize("changed", range(8), ids=lambda i: PARAMETERS[i])
def test_parameters_that_change_before_the_backward(calls, composed, changed, create_graph):
    """As with the separate operations: those that they save as they are
    raise, the others do not; a backward that is differentiated reads all of
    them and raises for each."""
    inputs = [t.requires_grad_(True) for t in _block_inputs(2, 6, 32, 4)]
    y = s4convd.S4BlockFused.apply(*inputs, 0.0)
    with torch.no_grad():
        inputs[1 + changed].add_(1.0)

    def backward():
        return torch.autograd.grad(y.sum(), inputs, create_graph=create_graph)

    if create_graph or PARAMETERS[changed] in ("c_re", "c_im", "a_im", "weight"):
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            backward()
    else:
        assert [g.shape for g in backward()] == [t.shape for t in inputs]
