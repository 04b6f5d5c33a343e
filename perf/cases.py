"""The cases the framework's speed is judged on: GroupNorm + activation as a user's program calls it, through GN_NHWC and
group_norm_nhwc, from the smallest call of a denoising step to tensors of half a gigabyte.

A case is a dict of plain values:
  mode      "infer" (forward without autograd) or "train" (forward, then the gradients of x, weight and bias)
  layout    "last" (channels-last memory, the framework's main path) or "first" (contiguous N, C, spatial)
  dtype     type of x;  params: type of weight and bias;  out: type y leaves in
  N, C, F, H, W, G   sizes; F > 0 makes the tensor 5-D (N, C, F, H, W)
  act       activation fused behind the normalisation
  add       True: y and s = x + residual + channel_bias[:, :, None, None] from one call (a ResNet block's second norm)
  offset    True: channels have their own means (as behind a convolution with a bias), False: N(0, 1)
"""
import math
import os
import sys

import torch

_PACKAGES = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "channels-last-groupnorm_amd")
if _PACKAGES not in sys.path:
    sys.path.insert(0, _PACKAGES)

from gnnhwc import GN_NHWC  # noqa: E402
from gnnhwc.custom_gn import group_norm_nhwc  # noqa: E402

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_BYTES = {"float32": 4, "float16": 2, "bfloat16": 2}
_ACTS = ("identity", "relu", "silu", "gelu", "gelu_tanh")

# The most bytes a drawn case may move (the largest listed one moves 1.07e9), and the most elements where the channel
# count is no multiple of a 16-byte vector or the layout is channels-first (such calls cost more per byte).
_MOST_BYTES = 8.0e8
_MOST_RAGGED = 2.0e7


def _case(name, mode, dtype, N, C, H, W, G, act, F=0, layout="last", params=None, out=None, add=False, offset=True):
    c = dict(mode=mode, layout=layout, dtype=dtype, params=params or dtype, out=out or dtype, N=N, C=C, F=F, H=H, W=W, G=G,
             act=act, add=add, offset=offset)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the deepest, smallest norm of a latent-diffusion UNet with two samples (guided denoising): latency only
        _case("unet_deep_infer_bf16", "infer", "bfloat16", 2, 1280, 8, 8, 32, "silu"),
        # one latent in full precision: the smallest benchmark configuration
        _case("unet_infer_f32", "infer", "float32", 1, 320, 64, 64, 32, "silu", offset=False),
        # a ResNet block's second norm in a denoising step: skip connection and time embedding added in the same call
        _case("resblock_add_infer_bf16", "infer", "bfloat16", 2, 640, 64, 64, 32, "silu", add=True),
        # fine-tuning at the middle UNet resolution
        _case("unet_train_f16", "train", "float16", 2, 640, 32, 32, 32, "silu", offset=False),
        # irregular image size: row counts that divide nothing
        _case("irregular_train_f32", "train", "float32", 3, 96, 37, 53, 24, "gelu", offset=False),
        # a channel count that is no multiple of the lane vector
        _case("ragged_channels_train_bf16", "train", "bfloat16", 6, 140, 64, 64, 4, "relu"),
        # 5-D (video) features on a float32 residual stream whose convolutions run in half precision
        _case("video_cast_train_f32", "train", "float32", 2, 256, 16, 16, 16, "gelu_tanh", F=8, out="bfloat16", offset=False),
        # the heaviest of the UNet benchmark shapes
        _case("unet_train_bf16", "train", "bfloat16", 4, 320, 128, 128, 32, "silu"),
        # the last blocks of an image decoder: few channels, many pixels
        _case("decoder_train_f16", "train", "float16", 1, 128, 512, 512, 32, "gelu_tanh", offset=False),
        # the same module on a tensor that was never brought into channels-last memory
        _case("channels_first_train_bf16", "train", "bfloat16", 1, 640, 128, 128, 32, "silu", layout="first"),
        # a training batch, float32 parameters beside half-precision activations as autocast leaves them
        _case("unet_batch_train_bf16", "train", "bfloat16", 16, 320, 128, 128, 32, "silu", params="float32"),
        # decoding a 1024 x 1024 image: the largest single tensor
        _case("decoder_infer_f16", "infer", "float16", 1, 256, 1024, 1024, 32, "silu", offset=False),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case: any mode, layout, type and activation of the listed ones, the size anywhere in their range (over its
    logarithm), image sizes and channels per group odd as often as not."""
    mode = rng.choice(("infer", "train", "train"))
    layout = "first" if rng.random() < 0.12 else "last"
    dtype = rng.choice(("float32", "float16", "bfloat16", "bfloat16"))
    act = rng.choice(_ACTS)
    ragged = rng.random() < 0.15
    vec = 16 // _BYTES[dtype]
    G = rng.choice((2, 4, 5) if ragged else (4, 8, 16, 24, 32, 32, 32))
    C = G * int(_log_uniform(rng, max(1, 16 // G), min(120, 2560 // G) + 1))
    if not ragged:  # groups as wide as it takes to fill whole vectors
        C = max(1, C // (G * vec)) * G * vec if C % vec else C
    elif C % vec == 0:
        C += G
        ragged = C % vec != 0
    add = layout == "last" and mode == "infer" and rng.random() < 0.3
    sizes = 5 if mode == "train" else 4 if add else 2
    most = _MOST_RAGGED if ragged or layout == "first" else _MOST_BYTES / (sizes * _BYTES[dtype])
    elements = _log_uniform(rng, 1.6e5, most)
    N = max(1, min(16, int(_log_uniform(rng, 1, 17))))
    while N > 1 and N * C * 9 > elements:
        N -= 1
    pixels = max(9.0, elements / (N * C))
    F = rng.choice((4, 5, 8)) if pixels >= 1024 and not add and rng.random() < 0.15 else 0
    side = math.sqrt(pixels / max(F, 1))
    H = max(3, int(side * rng.uniform(0.7, 1.0)))
    W = max(3, int(pixels / max(F, 1) / H))
    params = "float32" if dtype != "float32" and rng.random() < 0.25 else dtype
    out = rng.choice(("float16", "bfloat16")) if dtype == "float32" and layout == "last" and not add and rng.random() < 0.3 else dtype
    return _case(None, mode, dtype, N, C, H, W, G, act, F=F, layout=layout, params=params, out=out, add=add,
                 offset=rng.random() < 0.5)


def _spatial(case):
    return ((case["F"],) if case["F"] else ()) + (case["H"], case["W"])


def _activations(case, gen, dtype, offset):
    """(N, C, *spatial) in the case's layout."""
    N, C, spatial = case["N"], case["C"], _spatial(case)
    if case["layout"] == "first":
        t = torch.empty((N, C, *spatial), dtype=dtype, device="cuda").normal_(generator=gen)
        if offset:
            t.mul_(2.0).add_(torch.randn((C,) + (1,) * len(spatial), generator=gen, device="cuda").to(dtype))
        return t
    t = torch.empty((N, *spatial, C), dtype=dtype, device="cuda").normal_(generator=gen)
    if offset:
        t.mul_(2.0).add_(torch.randn((C,), generator=gen, device="cuda").to(dtype))
    return t.permute(0, t.dim() - 1, *range(1, t.dim() - 1))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, params, out = _DTYPES[case["dtype"]], _DTYPES[case["params"]], _DTYPES[case["out"]]
    m = GN_NHWC(case["G"], case["C"], activation=case["act"], out_dtype=out if out != dtype else None, device="cuda", dtype=params)
    with torch.no_grad():
        m.weight.uniform_(0.5, 1.5, generator=gen)
        m.bias.normal_(0.0, 0.1, generator=gen)
    state = dict(case=case, module=m, x=_activations(case, gen, dtype, case["offset"]))
    if case["add"]:
        state["residual"] = _activations(case, gen, dtype, False)
        state["channel_bias"] = torch.randn((case["N"], case["C"]), generator=gen, device="cuda").to(dtype)
    if case["mode"] == "train":
        state["x"].requires_grad_(True)
        state["dy"] = _activations(case, gen, out, False)
    return state


def run(state):
    case, m, x = state["case"], state["module"], state["x"]
    if case["mode"] == "train":
        y = m(x)
        dx, dweight, dbias = torch.autograd.grad(y, (x, m.weight, m.bias), state["dy"])
        return {"y": y.detach(), "dx": dx, "dweight": dweight, "dbias": dbias}
    with torch.no_grad():
        if case["add"]:
            y, s = group_norm_nhwc(x, m.weight, m.bias, case["G"], m.eps, case["act"], residual=state["residual"],
                                   channel_bias=state["channel_bias"], return_sum=True)
            return {"y": y, "sum": s}
        return {"y": m(x)}


def work(case):
    """The forward reads x and writes y; the backward, a later call of its own, reads x and dy and writes dx.  Operations per
    element: statistics 3, normalisation 2, activation 6; backward: 2 + 10 + 4 for the sums and 4 for dx."""
    elements = case["N"] * case["C"] * math.prod(_spatial(case))
    b, bo = _BYTES[case["dtype"]], _BYTES[case["out"]]
    nbytes, flops = elements * (b + bo), 11 * elements
    if case["add"]:  # the residual comes in, the sum goes out
        nbytes, flops = nbytes + 2 * elements * b, flops + 2 * elements
    if case["mode"] == "train":
        nbytes, flops = nbytes + elements * (2 * b + bo), flops + 20 * elements
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the outputs differ from the same path run in float64 on the same inputs: 2.4e-3 for bfloat16 (two
    roundings, g' and dx), 2.9e-4 for float16, 4e-7 for float32, 1.7e-3 where float32 data leaves as bfloat16.  relu's
    derivative jumps: a float32 element whose argument is zero to rounding may take either side (up to a few of 1e7)."""
    narrow = case["out"] if case["dtype"] == "float32" else case["dtype"]
    rel = {"float32": 2e-6, "float16": 1.2e-3, "bfloat16": 1e-2}[narrow]
    if case["act"] == "relu" and case["mode"] == "train":
        rel = max(rel, 3e-3)
    return {"rel": rel}


def _act64(name, t):
    if name == "identity":
        return t
    if name == "relu":
        return torch.relu(t)
    if name == "silu":
        return torch.nn.functional.silu(t)
    return torch.nn.functional.gelu(t, approximate="tanh" if name == "gelu_tanh" else "none")


def exact(case, seed):
    """The same outputs in float64 by plain torch, one sample at a time; dweight and dbias are summed over the samples."""
    state = prepare(case, seed)
    m, x = state["module"], state["x"].detach()
    C, G, N = case["C"], case["G"], case["N"]
    channels = (1, C) + (1,) * (x.dim() - 2)
    weight, bias = m.weight.detach().double().requires_grad_(True), m.bias.detach().double().requires_grad_(True)
    rows = {}

    def put(name, n, value):
        rows.setdefault(name, torch.empty(x.shape, dtype=torch.float64, device=x.device))[n:n + 1] = value

    dweight, dbias = torch.zeros_like(weight), torch.zeros_like(bias)
    for n in range(N):
        xn = x[n:n + 1].double()
        if case["add"]:
            xn = xn + state["residual"][n:n + 1].double() + state["channel_bias"][n].double().view(channels)
            put("sum", n, xn)
        xn.requires_grad_(case["mode"] == "train")
        with torch.set_grad_enabled(case["mode"] == "train"):
            groups = xn.reshape(1, G, -1)
            centred = groups - groups.mean(2, keepdim=True)
            xhat = (centred * torch.rsqrt(centred.square().mean(2, keepdim=True) + m.eps)).reshape(xn.shape)
            y = _act64(case["act"], xhat * weight.view(channels) + bias.view(channels))
        put("y", n, y.detach())
        if case["mode"] == "train":
            dx, dw, db = torch.autograd.grad(y, (xn, weight, bias), state["dy"][n:n + 1].double())
            put("dx", n, dx)
            dweight, dbias = dweight + dw, dbias + db
    if case["mode"] == "train":
        return {"y": rows["y"], "dx": rows["dx"], "dweight": dweight, "dbias": dbias}
    return rows
