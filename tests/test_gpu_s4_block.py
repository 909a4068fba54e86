"""The S4ConvD block's fused HIP passes (pt_s4_block_*) on the GPU (marked
``gpu``): output and every gradient against the same block in FP64 on the CPU
(the "pytorch" composition), over the channel counts, row lengths, state
counts and batch sizes where tiles end; and that every condition for running
the separate operations instead still gives the block's result.

Bar: 2e-6 of the tensor's 2-norm for outputs and input gradients (sums of up
to 512 products in FP32: sqrt(512) 2^-24 = 1.3e-6 for one rounding each at
random), 2e-5 for the parameters' (sums over all columns, and the taps'
gradients lose up to 1 / |dt A| through FP32 inputs of the chain)."""

from __future__ import annotations

import copy

import pytest
import torch

pytestmark = pytest.mark.gpu

ACT_TOL = 2e-6
PAR_TOL = 2e-5


@pytest.fixture(scope="module", autouse=True)
def rt():
    from pathtile_amd import runtime

    runtime.install_runtime(runtime.HipWarpRuntime())


def _rel(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return float((a - b).norm() / b.norm().clamp_min(1e-30))


def _make(B, H, L, state, p=0.0, seed=0):
    from pathtile_amd import s4convd

    torch.manual_seed(1000 + seed + B + H + L)
    block = s4convd.S4ConvBlock(H, state, p)
    x, gy = torch.randn(B, L, H), torch.randn(B, L, H)
    return block, x, gy


def _grads(block, x, gy):
    x = x.clone().requires_grad_(True)
    y = block(x)
    return [y, *torch.autograd.grad(y, (x, *block.parameters()), gy.to(y.dtype))]


def _fp64(block, x, gy):
    from pathtile_amd.kernels import warp_tiled_ampere as wta

    old, wta.TRAIN_CONV_BACKEND = wta.TRAIN_CONV_BACKEND, "pytorch"
    try:
        b = copy.deepcopy(block).cpu().double()
        # build_kernel's tap index is FP32; whole numbers, so exact in FP64 too
        return _grads(b, x.cpu().double(), gy.cpu().double())
    finally:
        wta.TRAIN_CONV_BACKEND = old


def _check(got, ref, names):
    for i, (a, b, n) in enumerate(zip(got, ref, names)):
        assert a.shape == b.shape, n
        assert _rel(a, b) < (ACT_TOL if i < 2 else PAR_TOL), (n, _rel(a, b))


@pytest.mark.parametrize("B,H,L,state", [
    (3, 32, 48, 64), (1, 32, 1, 2), (5, 64, 17, 16), (2, 64, 48, 70), (7, 96, 33, 32),
    (4, 128, 48, 64), (11, 128, 23, 64), (1, 128, 5, 6), (40, 128, 48, 64), (3, 160, 20, 16),
    (5, 192, 47, 32), (2, 224, 12, 8), (3, 256, 48, 64), (9, 256, 31, 18)])
def test_fused_block_against_fp64(B, H, L, state):
    print(f"[case] fused block B={B} H={H} L={L} state={state}", flush=True)
    block, x, gy = _make(B, H, L, state)
    names = ["y", "gx", *(n for n, _ in block.named_parameters())]
    ref = _fp64(block, x, gy)
    block.cuda()
    assert block._fused_inputs(x.cuda()) is not None
    got = _grads(block, x.cuda(), gy.cuda())
    _check(got, ref, names)
    again = _grads(block, x.cuda(), gy.cuda())
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    with torch.no_grad():
        assert torch.equal(block(x.cuda()), got[0])


def test_fused_block_many_tiles_per_workgroup():
    """More tiles than resident workgroups, and several 32-token steps per
    range of the weight gradient, against the separate operations."""
    block, x, gy = _make(3000, 64, 37, 16)
    block.cuda()
    got = _grads(block, x.cuda(), gy.cuda())
    block.activation.register_forward_hook(lambda *a: None)  # runs the separate operations
    assert block._fused_inputs(x.cuda()) is None
    with torch.backends.cudnn.flags(enabled=False):
        ref = _grads(block, x.cuda(), gy.cuda())
    names = ["y", "gx", *(n for n, _ in block.named_parameters())]
    _check(got, ref, names)


@pytest.mark.parametrize("B,H,L", [(33, 96, 29), (17, 32, 48), (5, 256, 36), (9, 160, 3)])
def test_fused_block_dropout_draws_the_modules_mask(B, H, L):
    """Training with dropout: the mask of the separate module under the same
    seed, in the output and the gradients (whole dwords of mask bytes and
    single ones)."""
    block, x, gy = _make(B, H, L, 16, p=0.3)
    block.cuda().train()
    torch.manual_seed(5)
    got = _grads(block, x.cuda(), gy.cuda())
    after = torch.cuda.get_rng_state()
    block.activation.register_forward_hook(lambda *a: None)
    torch.manual_seed(5)
    with torch.backends.cudnn.flags(enabled=False):
        ref = _grads(block, x.cuda(), gy.cuda())
    assert torch.equal(after, torch.cuda.get_rng_state())
    _check(got, ref, ["y", "gx", *(n for n, _ in block.named_parameters())])


def test_fused_block_partial_gradients():
    """Only what needs a gradient gets one, and it is the same."""
    block, x, gy = _make(6, 64, 48, 16)
    block.cuda()
    x, gy = x.cuda(), gy.cuda()
    full = dict(zip(["x", *(n for n, _ in block.named_parameters())], _grads(block, x, gy)[1:]))
    for keep in (["x"], ["output_linear.0.weight"], ["kernel_layer.C_re"], ["skip"]):
        for n, q in block.named_parameters():
            q.requires_grad_(n in keep)
            q.grad = None
        xi = x.clone().requires_grad_("x" in keep)
        block(xi).backward(gy)
        have = {n: q.grad for n, q in block.named_parameters() if q.grad is not None}
        if xi.grad is not None:
            have["x"] = xi.grad
        assert set(have) == set(keep)
        assert all(torch.equal(have[n], full[n]) for n in keep)


def test_fused_block_second_order_through_the_projection():
    """create_graph works as it does for the separate operations."""
    block, x, gy = _make(3, 32, 20, 8)
    block.cuda()
    x, gy = x.cuda(), gy.cuda()

    def second(b):
        y = b(x)
        w = b.output_linear[0].weight
        (g,) = torch.autograd.grad(y, w, gy, create_graph=True)
        return g, torch.autograd.grad(g.square().sum(), w)[0]

    with torch.backends.cudnn.flags(enabled=False):
        got = second(block)
        block.activation.register_forward_hook(lambda *a: None)
        ref = second(block)
    assert _rel(got[0], ref[0]) < PAR_TOL and _rel(got[1], ref[1]) < PAR_TOL


def test_fused_block_non_finite_values_stay_in_their_windows():
    """An Inf or NaN input reaches the tokens that the separate operations
    give it to, with the same kind of value, and no others."""
    block, x, gy = _make(4, 64, 24, 16)
    block.cuda()
    x, gy = x.cuda(), gy.cuda()
    x[1, 5, 3] = float("inf")
    x[2, 20, 7] = float("nan")
    gy[3, 2, 9] = float("inf")
    got = _grads(block, x, gy)
    block.activation.register_forward_hook(lambda *a: None)
    with torch.backends.cudnn.flags(enabled=False):
        ref = _grads(block, x, gy)
    for a, b in zip(got[:2], ref[:2]):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b))
        fine = torch.isfinite(b)
        assert _rel(a[fine], b[fine]) < 1e-5
    for a, b in zip(got[2:], ref[2:]):
        assert bool((torch.isfinite(a) == torch.isfinite(b)).all())


@pytest.mark.parametrize("log_a_re", [-50.0, -60.0])
def test_fused_block_poles_near_zero(log_a_re):
    """|A|^2 below FP32's range: the taps reach their limit 2 Re sum C dt, as
    they do to |dt A| L <= 3e-5 of it at A = -exp(-12)."""
    block, x, _ = _make(3, 32, 48, 16)
    block.cuda()
    out = []
    for a in (log_a_re, -12.0):
        with torch.no_grad():
            block.kernel_layer.log_A_re.fill_(a)
            block.kernel_layer.A_im.zero_()
            assert block._fused_inputs(x.cuda()) is not None
            out.append(block(x.cuda()))
    assert _rel(*out) < 1e-4


@pytest.mark.parametrize("how", ["hook", "collector", "strided", "autocast", "channels", "gelu"])
def test_separate_operations_still_serve(how):
    """Each condition that rules the fused passes out runs the separate
    operations, with the block's result."""
    from pathtile_amd.runtime import KERNEL_EVENTS

    H = 40 if how == "channels" else 64
    block, x, gy = _make(5, H, 16, 8)
    if how == "gelu":
        block.activation = torch.nn.GELU(approximate="tanh")
    ref = _fp64(block, x, gy)
    block.cuda()
    x = x.cuda()
    seen = []
    with torch.backends.cudnn.flags(enabled=False), \
            torch.autocast("cuda", torch.bfloat16, enabled=how == "autocast"):
        if how == "hook":
            block.output_linear[1].register_forward_hook(lambda m, i, o: seen.append(o.shape))
        if how == "strided":
            x = x.transpose(0, 1).contiguous().transpose(0, 1)
        KERNEL_EVENTS.enabled = how == "collector"
        try:
            assert block._fused_inputs(x) is None
            y = block(x)
        finally:
            phases = [r["phase"] for r in KERNEL_EVENTS.rows()]
            KERNEL_EVENTS.enabled = False
            KERNEL_EVENTS.clear()
    assert (how != "hook") or seen
    assert (how != "collector") or phases == ["fwd"]
    assert _rel(y, ref[0]) < (5e-2 if how == "autocast" else 1e-5)


def test_fused_block_on_a_side_stream_under_graph_capture():
    """The block's forward and backward in a captured graph, replayed with
    new inputs and eager work between the replays."""
    block, x, gy = _make(20, 64, 48, 16)
    block.cuda()
    xs, gys = x.cuda(), gy.cuda()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        _grads(block, xs, gys)  # first calls look up device attributes
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = _grads(block, xs, gys)
    for k in range(3):
        xs.copy_(x.cuda() + k)
        graph.replay()
        torch.cuda.synchronize()
        ref = _grads(block, xs, gys)
        assert all(torch.equal(a, b) for a, b in zip(out, ref)), k


@pytest.mark.parametrize("B,L,H,n_in,n_out", [(1, 1, 4, 1, 1), (3, 48, 128, 4, 1), (700, 5, 36, 8, 4),
                                              (1500, 12, 1024, 3, 2), (33, 30, 260, 7, 3)])
def test_model_ends_against_fp64(B, L, H, n_in, n_out):
    """Encoder and last-column decoder, output and gradients, against FP64;
    sums of up to B L products in FP32."""
    from pathtile_amd import s4convd

    print(f"[case] ends B={B} L={L} H={H} in={n_in} out={n_out}", flush=True)
    torch.manual_seed(B + H)
    enc, dec = torch.nn.Linear(n_in, H), torch.nn.Linear(H, n_out)
    x, gy = torch.randn(B, L, n_in), torch.randn(B, n_out)
    h, gh = torch.randn(B, L, H), torch.randn(B, L, H)

    def grads(dev, dtype, encode, head):
        e, d = copy.deepcopy(enc).to(dev, dtype), copy.deepcopy(dec).to(dev, dtype)
        xi, hi = (t.to(dev, dtype).requires_grad_(True) for t in (x, h))
        y, o = encode(e, xi), head(d, hi)
        return [y, o, *torch.autograd.grad(y, (xi, e.weight, e.bias), gh.to(dev, dtype)),
                *torch.autograd.grad(o, (hi, d.weight, d.bias), gy.to(dev, dtype))]

    ref = grads("cpu", torch.float64, lambda m, t: m(t), lambda m, t: m(t)[:, -1, :])
    got = grads("cuda", torch.float32,
                lambda m, t: s4convd.EncoderFused.apply(t, m.weight, m.bias),
                lambda m, t: s4convd.HeadFused.apply(t, m.weight, m.bias))
    for a, b in zip(got, ref):
        assert a.shape == b.shape and _rel(a, b) < 2e-6


def test_model_ends_follow_hooks_and_devices():
    """A hook on an end runs the module itself, with the same output."""
    from pathtile_amd import s4convd

    torch.manual_seed(3)
    m = s4convd.Model(state_dim=8, hidden_dim=32, input_dim=4, output_dim=2, num_blocks=1,
                      dropout=0.0).cuda()
    x = torch.randn(5, 12, 4, device="cuda")
    out, shapes = m(x), []
    for end in (m.encoder, m.decoder):
        end.register_forward_hook(lambda mod, i, o: shapes.append(tuple(o.shape)))
    with torch.backends.cudnn.flags(enabled=False):
        again = m(x)
    assert shapes == [(5, 12, 32), (5, 12, 2)]
    assert _rel(again, out) < 1e-6


@pytest.mark.parametrize("part", ["model", "block", "encoder"])
@pytest.mark.parametrize("how", ["strided", "half", "host"])
def test_saved_tensor_hooks_of_the_fused_functions(how, part):
    """What a hook unpacks reaches the kernels whole: strided copies give the
    same gradients, another type or device is refused."""
    from pathtile_amd import s4convd

    torch.manual_seed(5)
    model = s4convd.Model(state_dim=16, hidden_dim=64, num_blocks=1, dropout=0.1).cuda()
    x = torch.randn(33, 20, 64 if part == "block" else 4, device="cuda")
    if part == "block":
        part, model = model.blocks[0], model.blocks[0]
    elif part == "encoder":
        model = model.encoder
        part = lambda x: s4convd.EncoderFused.apply(x, model.weight, model.bias)  # noqa: E731
    else:
        part = model

    def unpack(t):
        if how == "strided":  # every second value of a buffer
            wide = torch.empty((*t.shape, 2), dtype=t.dtype, device=t.device)
            wide[..., 0] = t
            return wide[..., 0]
        return t.to(torch.float16) if how == "half" else t.cpu()

    def step(hooked):
        torch.manual_seed(6)
        if hooked:
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach().clone(), unpack):
                out = part(x)
        else:
            out = part(x)
        return torch.autograd.grad(out, tuple(model.parameters()), torch.ones_like(out))

    if how == "strided":  # the same kernels on the same values: the same bits
        assert all(torch.equal(a, b) for a, b in zip(step(True), step(False)))
    else:
        with pytest.raises(RuntimeError, match="was unpacked as"):
            step(True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float64])
def test_fused_model_under_another_default_dtype(dtype):
    """An FP32 model's step does not depend on torch's default dtype: the
    same bits."""
    from pathtile_amd import s4convd

    torch.manual_seed(8)
    model = s4convd.Model(state_dim=8, hidden_dim=64, output_dim=2, num_blocks=2,
                          dropout=0.1).cuda()
    x = torch.randn(17, 20, 4, device="cuda")

    def step():
        torch.manual_seed(9)
        out = model(x)
        return [out, *torch.autograd.grad(out, tuple(model.parameters()), torch.ones_like(out))]

    ref = step()
    old = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        got = step()
    finally:
        torch.set_default_dtype(old)
    for a, b in zip(got, ref):
        assert a.dtype == torch.float32 and torch.equal(a, b)


def test_fused_block_applied_twice_under_create_graph():
    """Gradients of a block that is applied to its own output, taken with
    create_graph: those of the separate operations."""
    block, x, gy = _make(3, 32, 20, 8)
    block.cuda()
    x, gy = x.cuda(), gy.cuda()
    inputs = (x.requires_grad_(True), *block.parameters())

    def grads():
        return torch.autograd.grad(block(block(x)), inputs, gy, create_graph=True)

    with torch.backends.cudnn.flags(enabled=False):
        got = grads()
        block.activation.register_forward_hook(lambda *a: None)
        ref = grads()
    for a, b in zip(got, ref):
        assert _rel(a, b) < PAR_TOL


@pytest.mark.parametrize("end", ["encoder", "decoder"])
@pytest.mark.parametrize("how", ["one bias", "more outputs"])
def test_model_ends_with_replaced_parameters(end, how):
    """A bias that ``F.linear`` broadcasts, and weights of other sizes than
    the module was made with, give the module's own result."""
    from pathtile_amd import s4convd

    torch.manual_seed(4)
    m = s4convd.Model(state_dim=8, hidden_dim=32, input_dim=4, output_dim=3, num_blocks=1,
                      dropout=0.0)
    lin = getattr(m, end)
    rows, width = lin.weight.shape
    if how == "one bias":
        lin.bias = torch.nn.Parameter(torch.randn(1))
    elif end == "decoder":
        lin.weight = torch.nn.Parameter(torch.randn(6, width))
        lin.bias = torch.nn.Parameter(torch.randn(6))
    else:  # and a block to match
        m.blocks[0] = s4convd.S4ConvBlock(64, 8, 0.0)
        m.decoder = torch.nn.Linear(64, 3)
        lin.weight = torch.nn.Parameter(torch.randn(64, width))
        lin.bias = torch.nn.Parameter(torch.randn(64))
    m.cuda()
    x = torch.randn(5, 12, 4, device="cuda")
    out = m(x)
    with torch.backends.cudnn.flags(enabled=False):
        ref = m.decoder(m.blocks[0](m.encoder(x)))[:, -1, :]
    assert out.shape == ref.shape and _rel(out, ref) < 1e-6


def test_model_compiles_to_one_graph_on_the_gpu():
    """The "pytorch" backend's composition as one graph of the compiler: the
    gate asks nothing of a GPU tensor that a compiler cannot trace."""
    from pathtile_amd import s4convd
    from pathtile_amd.kernels import warp_tiled_ampere as wta

    torch.manual_seed(6)
    m = s4convd.Model(state_dim=8, hidden_dim=32, num_blocks=2, dropout=0.0).cuda()
    x = torch.randn(3, 20, 4, device="cuda")
    old, wta.TRAIN_CONV_BACKEND = wta.TRAIN_CONV_BACKEND, "pytorch"
    try:
        with torch.backends.cudnn.flags(enabled=False), torch.no_grad():
            torch._dynamo.reset()
            assert _rel(torch.compile(m, fullgraph=True, backend="eager")(x), m(x)) < 1e-6
    finally:
        wta.TRAIN_CONV_BACKEND = old


def test_separate_launches_of_a_callers_runtime(monkeypatch):
    """A runtime that replaces the launches gets them from the block."""
    from pathtile_amd import runtime

    seen = []

    class Recording(runtime.HipWarpRuntime):
        def launch_fwd(self, *args, **kw):
            seen.append("fwd")
            super().launch_fwd(*args, **kw)

        def launch_bwd_input(self, *args, **kw):
            seen.append("dx")
            super().launch_bwd_input(*args, **kw)

        def launch_bwd_weight_deterministic(self, *args, **kw):
            seen.append("dk")
            super().launch_bwd_weight_deterministic(*args, **kw)

    block, x, gy = _make(5, 64, 16, 8)
    ref = _fp64(block, x, gy)
    block.cuda()
    monkeypatch.setattr(runtime, "_RUNTIME", Recording())
    with torch.backends.cudnn.flags(enabled=False):
        got = _grads(block, x.cuda(), gy.cuda())
    assert seen == ["fwd", "dx", "dk"]
    for a, b in zip(got, ref):
        assert _rel(a, b) < PAR_TOL


@pytest.mark.parametrize("how", ["PATHTILE_ROWS_ALGO", "PATHTILE_DK_ALGO", "rows_algo"])
def test_forced_kernel_choices_reach_the_blocks_launches(monkeypatch, how):
    """With a kernel named by the environment or the runtime the block runs
    the launches that follow it: the bits of the convolution's own function."""
    from pathtile_amd import runtime, s4convd

    block, x, gy = _make(40, 64, 48, 8)
    block.cuda()
    x = x.cuda()
    assert block._fused_inputs(x) is not None
    if how == "rows_algo":
        monkeypatch.setattr(runtime, "_RUNTIME", runtime.HipWarpRuntime(rows_algo="mfma"))
    else:
        monkeypatch.setenv(how, "valu")
    assert block._fused_inputs(x) is None
    seen = []
    block.dropout.register_forward_pre_hook(lambda m, i: seen.append(i[0]))
    with torch.backends.cudnn.flags(enabled=False):
        _grads(block, x, gy.cuda())
    k = block.kernel_layer.build_kernel(48, x.device)
    own = s4convd.depthwise_conv_skip_ampere(x.transpose(1, 2).contiguous(), k, block.skip)
    assert torch.equal(seen[0], own)


@pytest.mark.parametrize("how", ["is_grads_batched", "vmap"])
def test_batches_of_gradients_of_the_projection(how):
    """Batches of gradients where the separate operations take them: with the
    convolution's side frozen, against one gradient at a time."""
    block, x, gy = _make(3, 32, 20, 8)
    block.cuda()
    x, conv = x.cuda(), block.output_linear[0]
    for q in block.parameters():
        q.requires_grad_(q is conv.weight or q is conv.bias)
    y = block(x)
    gys = torch.stack([gy.cuda(), 2 - gy.cuda()])
    wrt = (conv.weight, conv.bias)
    with torch.backends.cudnn.flags(enabled=False):
        if how == "vmap":
            batch = torch.vmap(lambda g: torch.autograd.grad(y, wrt, g, retain_graph=True))(gys)
        else:
            batch = torch.autograd.grad(y, wrt, gys, is_grads_batched=True, retain_graph=True)
    for i in range(2):
        for a, b in zip(batch, torch.autograd.grad(y, wrt, gys[i], retain_graph=True)):
            assert _rel(a[i], b) < PAR_TOL


def test_fused_blocks_input_may_change_before_its_backward():
    block, x, gy = _make(4, 64, 24, 8)
    block.cuda()
    x, gy = x.cuda(), gy.cuda()

    def grads(change):
        h = x.clone()
        y = block(h)
        if change:
            h += y.detach()
        return torch.autograd.grad(y, tuple(block.parameters()), gy)

    assert all(torch.equal(a, b) for a, b in zip(grads(True), grads(False)))


def test_model_ends_partial_gradients():
    """Every choice of the gradients that are asked for gives the same values."""
    from pathtile_amd import s4convd

    torch.manual_seed(14)
    for fn, rows in ((s4convd.EncoderFused, 12), (s4convd.HeadFused, 3)):
        x, w, b = (torch.randn(*shape, device="cuda") for shape in ((9, 7, 8), (rows, 8), (rows,)))
        full = None
        for needs in range(7, 0, -1):
            ts = [t.clone().requires_grad_(bool(needs >> i & 1)) for i, t in enumerate((x, w, b))]
            out = fn.apply(*ts)
            g = iter(torch.autograd.grad(out, [t for t in ts if t.requires_grad], out.detach()))
            got = [next(g) if t.requires_grad else None for t in ts]
            full = full or got
            for a, c in zip(got, full):
                assert a is None or _rel(a, c) < 1e-6


@pytest.mark.parametrize("value", [float("inf"), -float("inf"), float("nan")])
def test_fused_block_kinds_of_non_finite_outputs(value):
    """An infinite skip term makes whole rows of values and gates infinite:
    every output is finite, an infinity of a sign, or NaN as it is for the
    separate operations."""
    block, x, _ = _make(4, 64, 24, 16)
    block.cuda()
    x = x.cuda()
    with torch.no_grad(), torch.backends.cudnn.flags(enabled=False):
        block.skip[5] = value
        got = block(x)
        block.activation.register_forward_hook(lambda *a: None)
        ref = block(x)
    for kind in (torch.isfinite, torch.isposinf, torch.isneginf, torch.isnan):
        assert torch.equal(kind(got), kind(ref)), kind.__name__


@pytest.mark.parametrize("name", ["skip", "kernel_layer.log_dt", "kernel_layer.log_A_re",
                                  "output_linear.0.bias"])
def test_fused_blocks_parameters_that_may_change_before_its_backward(name):
    """The gradients are those at the values that the forward saw."""
    block, x, gy = _make(4, 64, 24, 16)
    block.cuda()
    x, gy = x.cuda(), gy.cuda()
    ref = _grads(block, x, gy)[1:]
    y = block(x.requires_grad_(True))
    with torch.no_grad():
        block.get_parameter(name).add_(0.5)
    got = torch.autograd.grad(y, (x, *block.parameters()), gy)
    assert all(torch.equal(a, b) for a, b in zip(got, ref))
