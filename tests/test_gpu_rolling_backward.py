"""GPU tests of backward launches with more workgroups than fit the device at once (set by set, like the forwards of
test_gpu_rolling.py) against torch in float64: float32 parameters and float32 statistics, so that what the sums lose shows in
dgamma / dbeta and not in how they are stored."""
import ctypes

import pytest
import torch

from gnnhwc import _cabi
from tests.gpu_harness import cabi_bwd, cabi_fwd, err

pytestmark = pytest.mark.gpu

# N, R, C, G for 16-bit data (float32 takes half the channels: chunks are 128 bytes wide): one sample in sets of one chunk that
# take half the device (two-level exchange); sets of two and of three chunks, the last tile of one row or nearly full; groups of
# several chunks; a last chunk of 32 bytes; one group, i.e. a sample per set
SHAPES = [(1, 262144, 256, 32), (7, 16385, 640, 32), (3, 40000, 640, 8), (2, 24575, 1088, 4), (33, 16384, 272, 17), (6, 32768, 256, 1)]
DTYPES = [torch.bfloat16, torch.float16, torch.float32]


def _case(N, R, C, G, dtype, device):
    C = C // 2 if dtype == torch.float32 else C
    gen = torch.Generator(device=device).manual_seed(N + R + C)
    x = torch.empty((N, R, C), device=device, dtype=dtype).normal_(generator=gen).mul_(1.5).add_(
        torch.randn((C,), device=device, generator=gen).to(dtype))
    dy = torch.empty((N, R, C), device=device, dtype=dtype).normal_(generator=gen)
    w, b = torch.rand((C,), device=device, generator=gen) + 0.5, 0.1 * torch.randn((C,), device=device, generator=gen)
    _, mean, rstd = cabi_fwd(x, w, b, G, 1e-5, 2)
    return x, dy, w, b, mean, rstd


def _assert_set_by_set():
    out = (ctypes.c_int64 * 7)()
    _cabi.check(_cabi.lib.gnnhwc_debug_last_launch(out), "gnnhwc_debug_last_launch")
    assert out[0] >= 0 and _cabi.kernel_kind_names()[out[0]] == "fused_bwd", _cabi.last_launch()
    # one launch of more workgroups than two of these fit a CU
    assert out[4] == 1 and out[2] > 0 and out[5] > 512, _cabi.last_launch()
    return out[2]


def _roundings(x, act, window):
    """How often dx is rounded to the data type.  16-bit calls that a few launches could serve keep g' = dy act'(z) in packed form
    between the passes (a window of 16 rows of x, or 8), the others dy (12 rows); the identity's and relu's g' needs no rounding."""
    assert window in ((12,) if x.dtype == torch.float32 else (8, 16) if act < 2 else (8, 12, 16)), window
    return 2 if x.dtype != torch.float32 and act >= 2 and window != 12 else 1


def _derivative(act, z):
    if act == 0:
        return torch.ones_like(z)
    if act == 1:
        return (z > 0).to(z.dtype)
    z = z.detach().requires_grad_()
    f = {2: torch.nn.functional.silu, 3: torch.nn.functional.gelu, 4: lambda t: torch.nn.functional.gelu(t, approximate="tanh")}[act]
    return torch.autograd.grad(f(z).sum(), z)[0]


def _against_float64(x, dy, w, b, G, dx, dw, db, roundings, act=2, eps=1e-5):
    """dx: a rounding to the data type leaves an error spread evenly over a spacing, 1 / sqrt(12) of it in the 2-norm; a spacing is
    2^-7 (bfloat16) or 2^-10 (float16) of a value of mantissa 1 and half of that of one just below 2, so that the relative 2-norm
    lies between 0.144 and 0.289 spacings of 1, at 0.212 for normally distributed values.  The bar is 0.27, and sqrt(2) times that
    for two roundings (one: 1.66e-3 in bfloat16, two: 2.35e-3; float32: the sums' own rounding, 1e-6).  dgamma, dbeta: the float32
    bar, 1e-5 of the largest, and where they are stored in 16 bits half a spacing."""
    N, R, C = x.shape
    W, B = w.double(), b.double()
    DW, DB, off, size = torch.zeros_like(W), torch.zeros_like(W), 0.0, 0.0
    for n in range(N):
        t = x[n].double().view(R, G, C // G)
        mu = t.mean((0, 2), keepdim=True)
        rs = ((t - mu).square().mean((0, 2), keepdim=True) + eps).rsqrt()
        xh = ((t - mu) * rs).view(R, C)
        z = xh * W + B
        g = dy[n].double() * _derivative(act, z)
        DW += (g * xh).sum(0)
        DB += g.sum(0)
        gw, xg = (g * W).view(R, G, -1), xh.view(R, G, -1)
        want = (rs * (gw - gw.mean((0, 2), keepdim=True) - xg * (gw * xg).mean((0, 2), keepdim=True))).reshape(R, C)
        off += (dx[n].double() - want).square().sum().item()
        size += want.square().sum().item()
    spacing = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 0.0}
    assert (off / size) ** 0.5 <= roundings ** 0.5 * 0.27 * spacing[x.dtype] + 1e-6, ((off / size) ** 0.5, roundings)
    assert err(dw, DW) <= 1e-5 + spacing[w.dtype] / 2 and err(db, DB) <= 1e-5 + spacing[w.dtype] / 2


@pytest.mark.parametrize("N,R,C,G", SHAPES)
@pytest.mark.parametrize("dtype", DTYPES)
def test_against_float64(N, R, C, G, dtype, device):
    print("rolling backward", N, R, C, G, dtype, flush=True)
    x, dy, w, b, mean, rstd = _case(N, R, C, G, dtype, device)
    dx, dw, db = cabi_bwd(dy, x, w, b, mean, rstd, G, 2)
    _against_float64(x, dy, w, b, G, dx, dw, db, _roundings(x, 2, _assert_set_by_set()))
    again = cabi_bwd(dy, x, w, b, mean, rstd, G, 2)
    for s, t in zip((dx, dw, db), again):
        assert torch.equal(s, t)
    inplace = cabi_bwd(dy, x, w, b, mean, rstd, G, 2, dx=dy)
    for s, t in zip((dx, dw, db), inplace):
        assert torch.equal(s, t)


# One sample that no launch holds, in sets that leave the streaming kernels the only other choice, and a batch that few launches would
# fill badly: what dx loses with every activation, float32 parameters and parameters of the data's type; and the streaming
# kernels' own dx, which is rounded once, on the first.
@pytest.mark.parametrize("N,R,C,G,few", [(1, 131072, 320, 32, False), (3, 36000, 640, 8, True)])
@pytest.mark.parametrize("act", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("dtype,params", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32), (torch.float32, torch.float32)])
def test_every_activation_against_float64(N, R, C, G, few, act, dtype, params, device):
    print("rolling backward", N, R, C, G, act, dtype, params, flush=True)
    x, dy, w, b, _, _ = _case(N, R, C, G, dtype, device)
    w, b = w.to(params), b.to(params)
    _, mean, rstd = cabi_fwd(x, w, b, G, 1e-5, act)
    if act == 1:  # no gradient so near the kink that a float32 z may lie on its other side
        for n in range(N):
            mu, rs = (t[n].double().repeat_interleave(w.numel() // G) for t in (mean, rstd))
            dy[n][((x[n].double() - mu) * rs * w.double() + b.double()).abs() < 1e-4] = 0
    dx, dw, db = cabi_bwd(dy, x, w, b, mean, rstd, G, act)
    roundings = _roundings(x, act, _assert_set_by_set())
    assert roundings == (2 if few and act >= 2 and dtype != torch.float32 else 1)
    _against_float64(x, dy, w, b, G, dx, dw, db, roundings, act)
    if not few:
        before = _cabi.set_resident(False)
        try:
            dx, dw, db = cabi_bwd(dy, x, w, b, mean, rstd, G, act)
        finally:
            _cabi.set_resident(before)
        assert _cabi.last_launch() == "multi-launch"
        _against_float64(x, dy, w, b, G, dx, dw, db, 1, act)


# Batches on both sides of the line that dgamma / dbeta draw (as many row tiles in a sample as blocks of channels in a chunk; chunks
# of 128 bytes), with more sets than four launches hold.
@pytest.mark.parametrize("N,R,C,G,dtype", [(80, 15360, 128, 32, torch.bfloat16), (150, 7168, 64, 32, torch.float32)])
def test_samples_with_fewer_tiles_than_blocks_are_left_to_the_streaming_kernels(N, R, C, G, dtype, device):
    print("rolling backward, bound", N, R, C, G, dtype, flush=True)
    for rows in (R, R + 1):
        gen = torch.Generator(device=device).manual_seed(rows)
        x, dy = (torch.empty((N, rows, C), device=device, dtype=dtype).normal_(generator=gen) for _ in range(2))
        w, b = torch.rand((C,), device=device, generator=gen) + 0.5, 0.1 * torch.randn((C,), device=device, generator=gen)
        _, mean, rstd = cabi_fwd(x, w, b, G, 1e-5, 2)
        dx, dw, db = cabi_bwd(dy, x, w, b, mean, rstd, G, 2)
        if rows == R:
            assert _cabi.last_launch() == "multi-launch"
        else:
            assert _roundings(x, 2, _assert_set_by_set()) == 1
        _against_float64(x, dy, w, b, G, dx, dw, db, 1)


@pytest.mark.parametrize("N,R,C,G", [(7, 16385, 640, 32), (1, 262144, 256, 32)])
@pytest.mark.parametrize("spins", [-2, 0, 2])
def test_expired_waits_are_recovered(spins, N, R, C, G, device):
    x, dy, w, b, mean, rstd = _case(N, R, C, G, torch.bfloat16, device)
    _cabi.lib.gnnhwc_resident_status()
    before = _cabi.lib.gnnhwc_debug_set_spin_limit(spins)
    try:
        dx, dw, db = cabi_bwd(dy, x, w, b, mean, rstd, G, 2)
        torch.cuda.synchronize()
    finally:
        _cabi.lib.gnnhwc_debug_set_spin_limit(before)
    window = _assert_set_by_set()
    assert _cabi.lib.gnnhwc_resident_status() == 1 or spins != -2
    _against_float64(x, dy, w, b, G, dx, dw, db, _roundings(x, 2, window))


def test_replayed_graph(device):
    x, dy, w, b, mean, rstd = _case(7, 16385, 640, 32, torch.bfloat16, device)
    ws = torch.empty((_cabi.lib.gnnhwc_bwd_workspace_bytes(7, 16385, 640, 32, 3),), dtype=torch.uint8, device=device)
    dx = torch.empty_like(x)
    cabi_bwd(dy, x, w, b, mean, rstd, 32, 2, dx=dx, ws=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _, dw, db = cabi_bwd(dy, x, w, b, mean, rstd, 32, 2, dx=dx, ws=ws)
        _assert_set_by_set()
    for i in range(3):
        dy.add_(i)
        graph.replay()
        torch.cuda.synchronize()
        want = cabi_bwd(dy, x, w, b, mean, rstd, 32, 2)
        torch.cuda.synchronize()
        for s, t in zip((dx, dw, db), want):
            assert torch.equal(s, t)
