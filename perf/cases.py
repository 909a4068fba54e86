"""The work that this framework is timed on: sizes, inputs, one pass through
the public entry points, and what the results are compared with.

Six kinds of work, each as a user's program calls it:

``conv``         ``depthwise_conv_ampere``: FP32 rows of up to 48 columns and
                 48 taps, forward and backward (y, dX, dK), the layer that
                 the benchmark and the tuner are about.
``conv_bf16``    ``depthwise_conv_bf16``: the same with bfloat16 activations
                 and gradients (FP32 taps and dK).
``conv_long``    ``kernels.shared_l192.depthwise_conv_shared``: rows of up to
                 192 columns, forward and backward.
``channels_last`` ``launch_bwd_weight_channels_last``: the weight gradient of
                 ``[B, 1, L, H]`` tensors behind the Flash-DWC bridge.
``block``        one ``S4ConvBlock`` in training: output, input gradient and
                 every parameter's gradient.
``model``        the S4ConvD ``Model``: a training step (outputs and
                 gradients under the RMSLE loss) or inference (outputs).
"""

from __future__ import annotations

import math

import torch

from pathtile_amd import runtime, s4convd
from pathtile_amd.kernels import shared_l192
from pathtile_amd.kernels import warp_tiled_ampere as wta

HIDDEN = (32, 64, 96, 128, 192, 256)
STATES = (16, 32, 64)


def listed():
    return [
        # The fixed-seed plumbing check: the smallest call, all launch cost.
        dict(name="conv_tiny", kind="conv", B=64, H=16, L=48, K=48),
        # Ragged batch and rows with more taps than columns.
        dict(name="conv_edge", kind="conv", B=1000, H=96, L=37, K=48),
        # A channel count with no factor of two.
        dict(name="conv_odd_channels", kind="conv", B=2000, H=131, L=44, K=9),
        # The headline workload.
        dict(name="conv_primary", kind="conv", B=16384, H=128, L=48, K=48),
        # The short-filter workload: the most bytes of the short rows.
        dict(name="conv_short_taps", kind="conv", B=32768, H=256, L=48, K=4),
        # The headline workload with half the bytes.
        dict(name="conv_bf16", kind="conv_bf16", B=16384, H=128, L=48, K=48),
        # The long-row benchmark of the reference's L192 module.
        dict(name="conv_long_l192", kind="conv_long", B=16384, H=128, L=192, K=192),
        # Long rows of an ordinary size, ragged in every dimension.
        dict(name="conv_long_ragged", kind="conv_long", B=2100, H=96, L=100, K=37),
        # The bridge's weight gradient at the headline size.
        dict(name="channels_last_dk", kind="channels_last", B=16384, H=128, L=48, K=48),
        # One layer of the model on a batch of an ordinary size.
        dict(name="block_train", kind="block", B=2048, hidden=128, state=64, L=48, dropout=0.01),
        # A training step of the default model at the reference's batch.
        dict(name="model_train", kind="model", train=True, B=16384, hidden=128, state=64, L=48,
             blocks=4, dropout=0.01),
        # Serving a small batch with the default model.
        dict(name="model_infer", kind="model", train=False, B=64, hidden=128, state=64, L=48,
             blocks=4, dropout=0.01),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("conv", "conv", "conv", "conv_bf16", "conv_long", "channels_last",
                       "block", "model_train", "model_infer"))
    if kind == "conv":
        # any channel count, or one of the usual ones
        H = _log_int(rng, 16, 256) if rng.random() < 0.5 else rng.choice((16, 64, 96, 128, 256))
        return dict(kind=kind, B=_log_int(rng, 64, 32768), H=H, L=rng.randint(8, 48),
                    K=rng.randint(3, 48))
    if kind == "conv_bf16":
        return dict(kind=kind, B=_log_int(rng, 64, 32768), H=8 * rng.randint(2, 32),
                    L=4 * rng.randint(2, 12), K=rng.randint(3, 48))
    if kind == "conv_long":
        return dict(kind=kind, B=_log_int(rng, 64, 16384), H=_log_int(rng, 8, 128),
                    L=rng.randint(49, 192), K=rng.randint(5, 192))
    if kind == "channels_last":
        return dict(kind=kind, B=16 * _log_int(rng, 8, 1024), H=32 * rng.randint(1, 8),
                    L=rng.randint(8, 48), K=rng.randint(3, 48))
    hidden, state = rng.choice(HIDDEN), rng.choice(STATES)
    L, dropout = rng.randint(12, 48), rng.choice((0.0, 0.01, 0.1))
    if kind == "block":
        return dict(kind=kind, B=_log_int(rng, 32, 8192), hidden=hidden, state=state, L=L,
                    dropout=dropout)
    if kind == "model_train":
        return dict(kind="model", train=True, B=_log_int(rng, 64, 8192), hidden=hidden,
                    state=state, L=L, blocks=rng.randint(1, 4), dropout=dropout)
    return dict(kind="model", train=False, B=_log_int(rng, 1, 2048), hidden=hidden, state=state,
                L=L, blocks=rng.randint(1, 4), dropout=dropout)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _conv_inputs(case, seed):
    """x, dY ~ N(0, 1) and w ~ N(0, 1/K), the benchmark's distributions."""
    g = _generator(seed)
    B, H, L, K = (case[n] for n in "BHLK")
    shape = (B, 1, L, H) if case["kind"] == "channels_last" else (B, H, L)
    dtype = torch.bfloat16 if case["kind"] == "conv_bf16" else torch.float32
    x = torch.randn(shape, device="cuda", generator=g).to(dtype)
    gy = torch.randn(shape, device="cuda", generator=g).to(dtype)
    k = torch.randn((H, K), device="cuda", generator=g) / math.sqrt(K)
    return x, gy, k


def _fill_like_init(module, g):
    """The module's parameters drawn from its own initial distributions with
    the generator `g`: uniform within 1/sqrt(fan in) for the linear layers,
    log_dt uniform between log 0.001 and log 0.1, A_im ones, the rest N(0, 1)."""
    lo, hi = math.log(0.001), math.log(0.1)
    with torch.no_grad():
        for name, p in module.named_parameters():
            leaf = name.rsplit(".", 1)[-1]
            if leaf == "log_dt":
                p.copy_(torch.rand(p.shape, device="cuda", generator=g) * (hi - lo) + lo)
            elif leaf == "A_im":
                p.fill_(1.0)
            elif leaf in ("weight", "bias"):
                owner = module.get_submodule(name.rsplit(".", 1)[0])
                bound = 1.0 / math.sqrt(owner.weight.shape[1])
                p.copy_((torch.rand(p.shape, device="cuda", generator=g) * 2 - 1) * bound)
            else:
                p.copy_(torch.randn(p.shape, device="cuda", generator=g))
    return module


def _block(case, seed):
    g = _generator(seed)
    block = s4convd.S4ConvBlock(case["hidden"], case["state"], case["dropout"]).cuda().train()
    _fill_like_init(block, g)
    shape = (case["B"], case["L"], case["hidden"])
    x = torch.randn(shape, device="cuda", generator=g)
    gy = torch.randn(shape, device="cuda", generator=g)
    return block, x, gy


def _model(case, seed):
    g = _generator(seed)
    model = s4convd.Model(state_dim=case["state"], hidden_dim=case["hidden"],
                          num_blocks=case["blocks"], dropout=case["dropout"]).cuda()
    _fill_like_init(model, g).train(case["train"])
    x = torch.randn((case["B"], case["L"], 4), device="cuda", generator=g)
    target = torch.rand((case["B"], 1), device="cuda", generator=g)
    return model, x, target


def prepare(case, seed):
    runtime.get_or_create_runtime()
    kind = case["kind"]
    state = dict(kind=kind, seed=int(seed))
    if kind == "block":
        state["block"], x, state["gy"] = _block(case, seed)
        state["x"] = x.requires_grad_(True)
    elif kind == "model":
        state["model"], state["x"], state["target"] = _model(case, seed)
        state["train"] = case["train"]
    else:
        x, state["gy"], k = _conv_inputs(case, seed)
        if kind == "channels_last":
            state["x"] = x
            state["dw"] = torch.empty((1, case["K"], case["H"]), device="cuda")
        else:
            state["x"], state["k"] = x.requires_grad_(True), k.requires_grad_(True)
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
CONV = {
    "conv": lambda x, k: wta.depthwise_conv_ampere(x, k),
    "conv_bf16": lambda x, k: runtime.depthwise_conv_bf16(x, k),
    "conv_long": lambda x, k: shared_l192.depthwise_conv_shared(x, k),
}


def run(state):
    kind = state["kind"]
    if kind == "channels_last":
        rt = runtime.get_or_create_runtime()
        rt.launch_bwd_weight_channels_last(state["x"], state["gy"], state["dw"], zero_first=True)
        return state["dw"]
    if kind == "block":
        # a step that can be repeated draws its dropout masks from a seed of its own
        torch.manual_seed(state["seed"])
        block, x = state["block"], state["x"]
        y = block(x)
        return [y.detach(), *torch.autograd.grad(y, (x, *block.parameters()), state["gy"])]
    if kind == "model":
        model = state["model"]
        if not state["train"]:
            with torch.no_grad():
                return model(state["x"])
        torch.manual_seed(state["seed"])
        model.zero_grad(set_to_none=True)
        out = model(state["x"])
        loss = s4convd.rmsle(out, state["target"])
        loss.backward()
        return [out.detach(), loss.detach(), *(p.grad for p in model.parameters())]
    if kind == "conv_long":
        shared_l192.reset_timing_collectors()
    x, k = state["x"], state["k"]
    y = CONV[kind](x, k)
    return [y.detach(), *torch.autograd.grad(y, (x, k), state["gy"])]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _conv_flops(B, H, L, K):
    """Two operations for every product of a tap with an element of its row."""
    p = K // 2
    return 2 * B * H * sum(max(0, min(L, L - (j - p)) - max(0, p - j)) for j in range(K))


def work(case):
    kind, B, L = case["kind"], case["B"], case["L"]
    if kind in ("conv", "conv_bf16", "conv_long", "channels_last"):
        H, K = case["H"], case["K"]
        n, taps = B * H * L, 4 * H * K
        size = 2 if kind == "conv_bf16" else 4
        if kind == "channels_last":
            return {"bytes": 2 * n * size + taps, "flops": _conv_flops(B, H, L, K)}
        # forward: x, y; backward, a call of its own: dY, x, dX; taps twice and dK
        return {"bytes": 5 * n * size + 3 * taps, "flops": 3 * _conv_flops(B, H, L, K)}
    H = case["hidden"]
    n = B * H * L
    # the convolution, and the H to 2 H projection of every column
    layer = _conv_flops(B, H, L, L) + 2 * B * L * H * 2 * H
    weights = 4 * (2 * H * H + 2 * H + 2 * H * case["state"] + 2 * H)
    if kind == "block":
        # forward: x, y; backward: dY, x, dX
        return {"bytes": 4 * 5 * n + 3 * weights, "flops": 3 * layer}
    blocks = case["blocks"]
    ends = 4 * B * L * 4 + 4 * B
    flops = blocks * layer + 2 * B * L * 4 * H + 2 * B * H
    if not case["train"]:
        # activations of a layer can stay on the chip: weights, inputs, outputs
        return {"bytes": ends + blocks * weights, "flops": flops}
    # every block's input is written once and read again by its backward, and
    # the gradient that passes between two blocks is written and read
    return {"bytes": 2 * ends + blocks * (4 * 5 * n + 3 * weights), "flops": 3 * flops}


# ---------------------------------------------------------------------------
# What the results may differ by
# ---------------------------------------------------------------------------
def tolerance(case):
    """About four times the distance from `exact` measured for each kind (in
    brackets); the sums run over up to a million products."""
    kind = case["kind"]
    if kind == "conv_bf16":
        return {"rel": 1e-2}  # bfloat16 outputs [1.7e-3]
    if kind == "conv_long":
        return {"rel": 2e-5}  # dK of 16384 x 192 columns [5.3e-6]
    if kind == "block":
        return {"rel": 1e-5}  # [2e-6, the kernel's parameters]
    if kind == "model":
        # gradients through four blocks [1.4e-5]; outputs [1.4e-6]
        return {"rel": 1e-4 if case["train"] else 1e-5}
    return {"rel": 5e-6}  # 32-bit sums [1e-7 to 8e-7]


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _span(L, s):
    """Columns t with 0 <= t + s < L."""
    return max(0, -s), min(L, L - s)


class _Conv64(torch.autograd.Function):
    """y[t] = sum_j k[j] x[t + j - K // 2] per row, one tap at a time."""

    @staticmethod
    def forward(ctx, x, k):
        ctx.save_for_backward(x, k)
        return _fwd64(x, k)

    @staticmethod
    def backward(ctx, gy):
        x, k = ctx.saved_tensors
        return _dx64(gy, k), _dk64(gy, x, k.shape[1])


def _fwd64(x, k):
    L, K = x.shape[2], k.shape[1]
    y = torch.zeros_like(x, dtype=torch.float64)
    for j in range(K):
        s = j - K // 2
        lo, hi = _span(L, s)
        if lo < hi:
            y[:, :, lo:hi] += k[:, j, None] * x[:, :, lo + s:hi + s]
    return y


def _dx64(gy, k):
    L, K = gy.shape[2], k.shape[1]
    gx = torch.zeros_like(gy, dtype=torch.float64)
    for j in range(K):
        s = j - K // 2
        lo, hi = _span(L, s)
        if lo < hi:
            gx[:, :, lo + s:hi + s] += k[:, j, None] * gy[:, :, lo:hi]
    return gx


def _dk64(gy, x, K):
    H, L = x.shape[1:]
    gk = torch.zeros((H, K), dtype=torch.float64, device=x.device)
    for j in range(K):
        s = j - K // 2
        lo, hi = _span(L, s)
        if lo < hi:
            gk[:, j] = (gy[:, :, lo:hi] * x[:, :, lo + s:hi + s]).sum(dim=(0, 2))
    return gk


def _conv_exact(case, seed):
    x, gy, k = _conv_inputs(case, seed)
    k, K = k.double(), case["K"]
    rows = max(1, (1 << 26) // (case["H"] * case["L"]))  # samples at a time
    y, gx, gk = torch.empty(x.shape, dtype=torch.float64, device="cuda"), None, 0
    cl = case["kind"] == "channels_last"
    gx = None if cl else torch.empty_like(y)
    for b in range(0, case["B"], rows):
        xs, gs = x[b:b + rows].double(), gy[b:b + rows].double()
        if cl:
            xs, gs = (t[:, 0].transpose(1, 2).contiguous() for t in (xs, gs))
        else:
            y[b:b + rows] = _fwd64(xs, k)
            gx[b:b + rows] = _dx64(gs, k)
        gk = gk + _dk64(gs, xs, K)
    return gk.t().contiguous()[None] if cl else [y, gx, gk]


def _block64(p, x, dropout):
    """One block on `x` [B, L, H] from the parameters `p` (without prefix)."""
    B, L, H = x.shape
    dt = p["kernel_layer.log_dt"].exp()
    A = torch.complex(-p["kernel_layer.log_A_re"].exp(), p["kernel_layer.A_im"])
    C = torch.complex(p["kernel_layer.C_re"], p["kernel_layer.C_im"])
    dtA = A * dt[:, None]
    t = torch.arange(L, device=x.device, dtype=torch.float64)
    k = 2 * ((C * (dtA.exp() - 1) / A)[:, :, None] * torch.exp(dtA[:, :, None] * t)).sum(1).real
    rows = x.transpose(1, 2).contiguous()
    y = _Conv64.apply(rows, k) + rows * p["skip"][:, None]
    if dropout > 0:  # the same mask as for 32-bit values of this shape
        ones = torch.ones(y.shape, device=x.device)
        y = y * (torch.nn.functional.dropout(ones, dropout) != 0) / (1.0 - dropout)
    y = 0.5 * y * (1 + torch.erf(y / math.sqrt(2.0)))
    z = y.transpose(1, 2).reshape(B * L, H) @ p["output_linear.0.weight"][:, :, 0].t()
    z = z + p["output_linear.0.bias"]
    return (z[:, :H] * torch.sigmoid(z[:, H:])).reshape(B, L, H) + x


def _params64(module):
    return {n: p.detach().double().requires_grad_(True) for n, p in module.named_parameters()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "block":
        block, x, gy = _block(case, seed)
        p = _params64(block)
        x = x.double().requires_grad_(True)
        torch.manual_seed(int(seed))
        y = _block64(p, x, case["dropout"])
        return [y.detach(), *torch.autograd.grad(y, (x, *p.values()), gy.double())]
    if kind == "model":
        model, x, target = _model(case, seed)
        p, train = _params64(model), case["train"]
        torch.manual_seed(int(seed))
        with torch.set_grad_enabled(train):
            h = x.double() @ p["encoder.weight"].t() + p["encoder.bias"]
            for i in range(case["blocks"]):
                head = "blocks.%d." % i
                one = {n[len(head):]: v for n, v in p.items() if n.startswith(head)}
                h = _block64(one, h, case["dropout"] if train else 0.0)
            out = h[:, -1] @ p["decoder.weight"].t() + p["decoder.bias"]
            if not train:
                return out
            a, b = out.reshape(-1).clamp(min=0), target.double().reshape(-1)
            loss = torch.sqrt((a.log1p() - b.log1p()).square().mean() + 1e-12)
            return [out.detach(), loss.detach(), *torch.autograd.grad(loss, tuple(p.values()))]
    return _conv_exact(case, seed)
