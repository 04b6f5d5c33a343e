"""GPU tests of the streaming kernels at the sizes where their work is cut differently: C ABI calls with the single-launch
kernels switched off, against torch in float64 with the bars of tests/test_gpu_parity.py."""
import pytest
import torch

from gnnhwc import _cabi
from tests.gpu_harness import cabi_bwd, cabi_fwd, err, far_from_zero
from tests.test_gpu_parity import FP32_TOL, _check_against_torch

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def streaming_only():
    before = _cabi.set_resident(False)
    yield
    _cabi.set_resident(before)


# dgamma / dbeta are summed over N * tiles entries by 32, 16 or 8 channels per workgroup (up to 64, 128, more entries), the
# pieces of a chunk handed out over the samples: channel counts below, at and beside those widths, chunks that are one piece
# and many, more samples than pieces and fewer, entries below the lanes of a channel.
@pytest.mark.parametrize("N,R,C,G", [(1, 7, 3, 1), (1, 40, 31, 1), (2, 65, 33, 3), (1, 300, 7, 7), (5, 1000, 35, 5),
                                     (6, 4096, 140, 4), (1, 30000, 70, 2), (3, 9000, 257, 1), (40, 9, 66, 2), (4, 3000, 64, 8),
                                     (1, 20000, 320, 32)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_parameter_gradients_of_the_streaming_backward(N, R, C, G, dtype, device):
    print("streaming", N, R, C, G, dtype, flush=True)
    _check_against_torch(N, R, C, G, "silu", dtype, device)
    assert _cabi.last_launch() == "multi-launch"


# Lane vectors of 16, 8, 4 and 2 bytes (f32: 16, 8, 4): what the channel count divides, and what the addresses divide (the
# tensors are cut out of larger buffers `shift` elements in).  Few and many channels, chunks of a whole row and of less.
@pytest.mark.parametrize("C,G", [(4, 2), (12, 3), (36, 4), (140, 4), (1100, 4), (6, 1), (70, 2), (2050, 5), (35, 5), (64, 8)])
@pytest.mark.parametrize("shift", [0, 1, 2, 4])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
def test_lane_vector_widths(C, G, shift, dtype, device):
    N, R = 2, 67
    gen = torch.Generator().manual_seed(C * 10 + shift)

    def cut(t):
        buf = torch.empty(t.numel() + 16, dtype=dtype, device=device)
        out = buf[shift:shift + t.numel()].view(t.shape)
        out.copy_(t)
        return out

    x, dy = (cut(torch.randn((N, R, C), generator=gen).to(dtype)) for _ in range(2))
    w, b = torch.rand(C, generator=gen).to(dtype).to(device) + 0.5, torch.randn(C, generator=gen).to(dtype).to(device)
    want = dtype if dtype == torch.float64 else torch.float32
    eps = {torch.float32: 1e-5, torch.float64: 1e-12, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]  # two spacings
    xt, wt, bt = x.to(want).permute(0, 2, 1).requires_grad_(), w.to(want).requires_grad_(), b.to(want).requires_grad_()
    yt = torch.nn.functional.silu(torch.nn.functional.group_norm(xt.contiguous(), G, wt, bt, 1e-5))
    gx, gw, gb = torch.autograd.grad(yt, (xt, wt, bt), dy.to(want).permute(0, 2, 1))
    y, mean, rstd = cabi_fwd(x, w, b, G, 1e-5, 2, y=cut(torch.zeros(N, R, C)))
    dx, dw, db = cabi_bwd(dy, x, w, b, mean, rstd, G, 2, dx=cut(torch.zeros(N, R, C)))
    for a, t in ((y, yt.permute(0, 2, 1)), (dx, gx.permute(0, 2, 1)), (dw, gw), (db, gb)):
        assert err(a, t) <= eps, (err(a, t), eps)


# The consumers' own tiling: rows that widen to 16, 32, 64 and 128 lane vectors or stay, with and without the compaction launch,
# more groups than a widened row may have, a row count of one tile, one row more, and one row less than whole tiles.
@pytest.mark.parametrize("N,R,C,G", [(1, 8192, 128, 32), (2, 8193, 256, 8), (1, 65535, 512, 64), (1, 4097, 1024, 128),
                                     (1, 4096, 1024, 512), (3, 2047, 320, 32), (1, 70001, 64, 1), (2, 513, 2048, 4)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_consumer_tiling(N, R, C, G, dtype, device):
    print("consumer tiling", N, R, C, G, dtype, flush=True)
    _check_against_torch(N, R, C, G, "gelu_tanh", dtype, device)
    assert _cabi.last_launch() == "multi-launch"


# The statistics pass takes every tiles-th batch of eight rows per lane: fewer rows per lane than a batch (1, 2, 4, 5, 7), one batch
# and a part of one, as many batches as tiles, one row more and less than whole batches, several samples, more samples than a
# grid has layers; and tensors beyond what the memory-side cache is counted on to hold (the last four), whose first batches and
# whose consumer use non-temporal loads.  One mean for all channels, many standard deviations away, and one row further off
# still: sums about anything but a value of the data lose what test_oracle.py's test of lane sums shows.  FP32_TOL is the bar of
# all float32 results; y = x a + c adds half a spacing of its type and, of x a, the roundings of a, of the mean and of c.
@pytest.mark.parametrize("N,R,C,G,dtype", [
    (1, 1, 64, 8, torch.float32), (2, 255, 64, 8, torch.float32), (2, 257, 64, 8, torch.bfloat16), (1, 16384 * 12, 64, 2, torch.float32),
    (300, 32, 64, 8, torch.bfloat16), (300, 64, 64, 8, torch.float16), (400, 128, 64, 8, torch.bfloat16), (500, 160, 64, 8, torch.float16),
    (500, 225, 64, 8, torch.bfloat16), (65537, 33, 16, 2, torch.bfloat16),
    (1, 16384 * 12 + 1, 64, 2, torch.float16), (3, 16384 * 4 - 1, 64, 8, torch.float32), (1, 7919, 140, 4, torch.bfloat16),
    (2, 40007, 64, 8, torch.float64), (1, 940007, 64, 8, torch.float32), (3, 170003, 128, 16, torch.float32),
    (1, 524287, 256, 32, torch.float16), (2, 262145, 256, 8, torch.bfloat16)])
def test_statistics_of_swept_rows(N, R, C, G, dtype, device):
    print("swept rows", N, R, C, G, dtype, flush=True)
    gen = torch.Generator(device=device).manual_seed(R + C)
    x = torch.empty((N, R, C), dtype=dtype, device=device)
    for n in range(0, N, 4096):
        x[n:n + 4096] = far_from_zero(min(4096, N - n), R, C, dtype, gen)
    w, b = torch.rand(C, generator=gen, device=device).to(dtype) + 0.5, torch.randn(C, generator=gen, device=device).to(dtype)
    y, mean, rstd = cabi_fwd(x, w, b, G, 1e-5, 0)
    assert _cabi.last_launch() == "multi-launch"
    half = {torch.float32: 0.0, torch.float64: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    for n in range(N) if N < 8 else (0, 1, N // 2, N - 1):
        xd = x[n].double().view(R, G, C // G)
        mu, var = xd.mean(dim=(0, 2)), xd.var(dim=(0, 2), correction=0)
        rs = (var + 1e-5).rsqrt()
        assert err(mean[n], mu) <= FP32_TOL and err(rstd[n], rs) <= FP32_TOL, (err(mean[n], mu), err(rstd[n], rs))
        xa = xd * rs[:, None]
        want = (xa - (mu * rs)[:, None]).view(R, C) * w.double() + b.double()
        off = (y[n].double() - want).abs() / (want.abs() + want.square().mean().sqrt() + 1e-30)
        lost = 4 * 2.0 ** -24 * float((xa.abs().view(R, C) * w.double()).max() / want.square().mean().sqrt())
        assert float(off.max()) <= FP32_TOL + half + (0.0 if dtype == torch.float64 else lost), float(off.max())


@pytest.mark.parametrize("want_dw,want_db", [(True, False), (False, True), (False, False)])
def test_parameter_gradients_not_asked_for(want_dw, want_db, device):
    x, dy = torch.randn(3, 500, 35, device=device), torch.randn(3, 500, 35, device=device)
    w, b = torch.rand(35, device=device) + 0.5, torch.randn(35, device=device)
    _, mean, rstd = cabi_fwd(x, w, b, 5, 1e-5, 2)
    dx, dw, db = cabi_bwd(dy, x, w, b, mean, rstd, 5, 2)
    dx2, dw2, db2 = cabi_bwd(dy, x, w, b, mean, rstd, 5, 2, want_dw=want_dw, want_db=want_db)
    assert torch.equal(dx, dx2)
    assert torch.equal(dw, dw2) if want_dw else dw2 is None
    assert torch.equal(db, db2) if want_db else db2 is None
