"""GPU tests of forward launches with more workgroups than fit the device at once: sets of workgroups that exchange records
follow each other through it.  Against torch in float64 and against the streaming kernels on the same inputs: statistics
agree to float32 rounding, y to that or to one spacing of its 16-bit type."""
import ctypes

import pytest
import torch

from gnnhwc import _cabi
from tests.gpu_harness import cabi_fwd, cabi_fwd_add, err

pytestmark = pytest.mark.gpu

# N, R, C, G: sets of one chunk (groups inside a chunk; several in flight, and one that takes half the device), of two and three
# chunks (groups across chunk borders), of a whole sample (one group), a last tile of one row, of all but one, chunks of 32 bytes
SHAPES = [(7, 16384, 320, 32), (1, 262144, 192, 12), (2, 65537, 256, 32), (3, 40000, 640, 8), (70, 513, 1280, 32), (2, 24575, 1088, 4),
          (6, 32768, 256, 1), (9, 16384, 272, 17)]


def _inputs(N, R, C, dtype, device):
    gen = torch.Generator(device=device).manual_seed(N + R + C)
    x = torch.empty((N, R, C), device=device, dtype=dtype).normal_(generator=gen).mul_(1.5).add_(
        torch.randn((C,), device=device, generator=gen).to(dtype))
    w = (torch.rand((C,), device=device, generator=gen) + 0.5).to(dtype)
    b = (0.1 * torch.randn((C,), device=device, generator=gen)).to(dtype)
    return x, w, b


def _close(y, y0, mean, mean0, rstd, rstd0):
    # float32 statistics of up to 1e8 elements, summed in two orders
    assert (mean - mean0).abs().max() <= 2e-6
    assert ((rstd - rstd0).abs() / rstd0).max() <= 2e-6
    eps = torch.finfo(y.dtype).eps  # one spacing is eps |y| at most; a statistic's rounding moves y by about 1e-6
    for n in range(y.shape[0]):
        a, t = y[n].float(), y0[n].float()
        assert ((a - t).abs() <= (eps if y.dtype != torch.float32 else 0) * t.abs() + 1e-5).all()


def _assert_set_by_set(x, kernel="fused_fwd"):
    """The last call was one launch of a single-launch kernel on more than the 64 MiB that such a launch can hold in
    registers (512 workgroups of 32 rows per lane, or 1024 of 16): its workgroups were not all resident at once."""
    out = (ctypes.c_int64 * 7)()
    _cabi.check(_cabi.lib.gnnhwc_debug_last_launch(out), "gnnhwc_debug_last_launch")
    assert out[0] >= 0 and _cabi.kernel_kind_names()[out[0]] == kernel, _cabi.last_launch()
    rows, workgroups = int(out[1]), int(out[5])
    assert out[4] == 1 and x.numel() * x.element_size() > 64 << 20
    assert workgroups > (512 if rows == 32 else 1024), (rows, workgroups)


def _against_float64(x, w, b, G, y, mean, rstd, eps=1e-5, act=2):
    """y = silu (act 3: gelu) of normalised x: within one rounding to its type of a value that meets the float32 bar (1e-5)."""
    N, R, C = x.shape
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[x.dtype]
    for n in range(N):
        t = x[n].double().view(R, G, C // G)
        mu = t.mean((0, 2), keepdim=True)
        var = (t - mu).square().mean((0, 2), keepdim=True)
        rs = (var + eps).rsqrt()
        assert err(mean[n], mu) <= 1e-5 and err(rstd[n], rs) <= 1e-5
        f = torch.nn.functional.gelu if act == 3 else torch.nn.functional.silu
        z = f(((t - mu) * rs).view(R, C) * w.double() + b.double())
        assert bool(((y[n].double() - z).abs() <= half * z.abs() * 1.001 + 1e-5 * (z.abs() + 1.0)).all())


def _streaming(fn):
    before = _cabi.set_resident(False)
    try:
        return fn()
    finally:
        _cabi.set_resident(before)


@pytest.mark.parametrize("N,R,C,G", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_against_float64_and_the_streaming_kernels(N, R, C, G, dtype, device):
    print("rolling", N, R, C, G, dtype, flush=True)
    x, w, b = _inputs(N, R, C, dtype, device)
    y, mean, rstd = cabi_fwd(x, w, b, G, 1e-5, 2)
    _assert_set_by_set(x)
    _against_float64(x, w, b, G, y, mean, rstd)
    again = cabi_fwd(x, w, b, G, 1e-5, 2)
    for s, t in zip((y, mean, rstd), again):
        assert torch.equal(s, t)
    del again
    y0, mean0, rstd0 = _streaming(lambda: cabi_fwd(x, w, b, G, 1e-5, 2))
    _close(y, y0, mean, mean0, rstd, rstd0)
    inplace = cabi_fwd(x, w, b, G, 1e-5, 2, y=x)[0]
    assert torch.equal(inplace, y)


# Both sides of the lines between 16 and 32 rows per lane (256 CUs): workgroups of 16 rows beyond 4/3 of the 1024 resident ones, where
# all poll all; tiles of a sample below and from 18 on; groups that are merged in two levels whatever the workgroups; 16-bit gelu.
@pytest.mark.parametrize("N,R,C,G,dtype,act,rows", [
    (2, 43520, 256, 16, torch.float32, 2, 16), (2, 43521, 256, 16, torch.float32, 2, 32), (6, 21500, 320, 32, torch.bfloat16, 2, 16),
    (16, 16384, 320, 32, torch.bfloat16, 2, 32), (24, 8704, 320, 32, torch.float16, 2, 16), (24, 8705, 320, 32, torch.float16, 2, 32),
    (4, 65536, 128, 32, torch.float32, 2, 16), (16, 16384, 320, 32, torch.bfloat16, 3, 16), (2, 43521, 256, 16, torch.float32, 3, 32)])
def test_rows_per_lane(N, R, C, G, dtype, act, rows, device):
    print("rolling rows", N, R, C, G, dtype, act, flush=True)
    x, w, b = _inputs(N, R, C, dtype, device)
    y, mean, rstd = cabi_fwd(x, w, b, G, 1e-5, act)
    _assert_set_by_set(x)
    assert "rows=%d " % rows in _cabi.last_launch(), _cabi.last_launch()
    _against_float64(x, w, b, G, y, mean, rstd, act=act)


# The same for launches that are resident as a whole: more than 768 workgroups of 16 rows that all poll more than 900 records (980;
# 588 in wider groups; 720 workgroups; two levels).
@pytest.mark.parametrize("N,R,C,G,dtype,rows", [(1, 50000, 256, 32, torch.float32, 32), (1, 50000, 256, 16, torch.float32, 16),
                                                (1, 46000, 256, 32, torch.float32, 16), (1, 60000, 512, 32, torch.bfloat16, 16)])
def test_rows_per_lane_of_one_resident_launch(N, R, C, G, dtype, rows, device):
    x, w, b = _inputs(N, R, C, dtype, device)
    y, mean, rstd = cabi_fwd(x, w, b, G, 1e-5, 2)
    assert _cabi.last_launch().startswith("fused_fwd rows=%d " % rows), _cabi.last_launch()
    _against_float64(x, w, b, G, y, mean, rstd)
    s, mean, rstd = (t for i, t in enumerate(cabi_fwd_add(x, None, torch.zeros(N, C, device=device, dtype=dtype), w, b, G, 1e-5, 2)) if i != 1)
    assert _cabi.last_launch().startswith("fused_fwd_add rows=%d " % rows), _cabi.last_launch()
    _against_float64(x, w, b, G, s, mean, rstd)


def test_with_fused_additions(device):
    x, w, b = _inputs(9, 16384, 320, torch.bfloat16, device)
    r, cb = torch.randn_like(x), torch.randn(9, 320, device=device).bfloat16()
    y, s, mean, rstd = cabi_fwd_add(x, r, cb, w, b, 32, 1e-5, 2)
    _assert_set_by_set(x, "fused_fwd_add")
    _against_float64(s, w, b, 32, y, mean, rstd)
    y0, s0, mean0, rstd0 = _streaming(lambda: cabi_fwd_add(x, r, cb, w, b, 32, 1e-5, 2))
    assert torch.equal(s, s0)
    _close(y, y0, mean, mean0, rstd, rstd0)


# The all-to-all exchange, and the two-level one (one row of the last tile; groups in the middle of chunks and across them).
@pytest.mark.parametrize("N,R,C,G", [(14, 16384, 160, 16), (2, 65537, 256, 32)])
@pytest.mark.parametrize("spins", [-2, 0, 2])
def test_expired_waits_are_recovered(spins, N, R, C, G, device):
    x, w, b = _inputs(N, R, C, torch.bfloat16, device)
    y0, mean0, rstd0 = _streaming(lambda: cabi_fwd(x, w, b, G, 1e-5, 2))
    _cabi.lib.gnnhwc_resident_status()
    before = _cabi.lib.gnnhwc_debug_set_spin_limit(spins)
    try:
        y, mean, rstd = cabi_fwd(x, w, b, G, 1e-5, 2)
        torch.cuda.synchronize()
    finally:
        _cabi.lib.gnnhwc_debug_set_spin_limit(before)
    _assert_set_by_set(x)
    assert ("two_level=1" in _cabi.last_launch()) == (G == 32)
    expired = _cabi.lib.gnnhwc_resident_status()
    assert expired == 1 or spins != -2
    _close(y, y0, mean, mean0, rstd, rstd0)
    _against_float64(x, w, b, G, y, mean, rstd)
    if spins == -2:
        return  # (recomputes records whose workgroups may have stored already: out of place only)
    before = _cabi.lib.gnnhwc_debug_set_spin_limit(spins)
    try:
        y, mean, rstd = cabi_fwd(x, w, b, G, 1e-5, 2, y=x)
        torch.cuda.synchronize()
    finally:
        _cabi.lib.gnnhwc_debug_set_spin_limit(before)
    _cabi.lib.gnnhwc_resident_status()
    _close(y, y0, mean, mean0, rstd, rstd0)


@pytest.mark.parametrize("R,G", [(16384, 32), (65537, 32)])
@pytest.mark.parametrize("spins", [-2, 2])
def test_expired_waits_with_fused_additions(spins, R, G, device):
    N, C = (9, 320) if R == 16384 else (2, 256)
    x, w, b = _inputs(N, R, C, torch.bfloat16, device)
    r, cb = torch.randn_like(x), torch.randn(N, C, device=device).bfloat16()
    y0, s0, mean0, rstd0 = _streaming(lambda: cabi_fwd_add(x, r, cb, w, b, G, 1e-5, 2))
    _cabi.lib.gnnhwc_resident_status()
    before = _cabi.lib.gnnhwc_debug_set_spin_limit(spins)
    try:
        y, s, mean, rstd = cabi_fwd_add(x, r, cb, w, b, G, 1e-5, 2)
        torch.cuda.synchronize()
    finally:
        _cabi.lib.gnnhwc_debug_set_spin_limit(before)
    _assert_set_by_set(x, "fused_fwd_add")
    expired = _cabi.lib.gnnhwc_resident_status()
    assert expired == 1 or spins != -2
    assert torch.equal(s, s0)
    _close(y, y0, mean, mean0, rstd, rstd0)


def test_replayed_graph(device):
    x, w, b = _inputs(8, 16384, 320, torch.bfloat16, device)
    ws = torch.empty((_cabi.lib.gnnhwc_fwd_workspace_bytes(8, 16384, 320, 32, 3),), dtype=torch.uint8, device=device)
    y = torch.empty_like(x)
    cabi_fwd(x, w, b, 32, 1e-5, 2, y=y, ws=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        cabi_fwd(x, w, b, 32, 1e-5, 2, y=y, ws=ws)
        _assert_set_by_set(x)
    for i in range(3):
        x.add_(i)
        graph.replay()
        torch.cuda.synchronize()
        want = cabi_fwd(x, w, b, 32, 1e-5, 2)[0]
        torch.cuda.synchronize()
        assert torch.equal(y, want)


# One row more than half the device holds, and sets of two and of four chunks beyond it: such a launch would have to have the
# device to itself, so the streaming kernels take these calls.
@pytest.mark.parametrize("N,R,C,G", [(1, 262145, 192, 12), (1, 524288, 192, 12), (1, 131073, 320, 32), (2, 65537, 256, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_sets_beyond_half_the_device_are_streamed(N, R, C, G, dtype, device):
    C = C // 2 if dtype == torch.float32 and C != 320 else C  # chunks are 128 bytes wide
    x, w, b = _inputs(N, R, C, dtype, device)
    cabi_fwd(x, w, b, G, 1e-5, 2)
    assert _cabi.last_launch() == "multi-launch"
    cabi_fwd_add(x, None, torch.zeros(N, C, device=device, dtype=dtype), w, b, G, 1e-5, 2)
    assert _cabi.last_launch() == "multi-launch"


def _beside(tenant, x, w, b, x2, w2, b2):
    streams = [torch.cuda.Stream() for _ in range(2)]
    want = [cabi_fwd(x, w, b, 32, 1e-5, 2), cabi_fwd(x2, w2, b2, 32, 1e-5, 2)]
    torch.cuda.synchronize()
    _cabi.lib.gnnhwc_resident_status()
    for stream in streams:
        with torch.cuda.stream(stream):
            tenant()
    got = [cabi_fwd(x, w, b, 32, 1e-5, 2), cabi_fwd(x2, w2, b2, 32, 1e-5, 2)]
    torch.cuda.current_stream().synchronize()
    print("tenants still there at the end:", [not stream.query() for stream in streams], flush=True)
    torch.cuda.synchronize()
    return want, got, _cabi.lib.gnnhwc_resident_status()


def test_beside_kernels_that_hold_a_few_places(device):
    """Kernels of other streams hold a place of the device each for as long as the launches below take many times over: the
    largest set there is becomes resident beside them, no wait expires, and the results are those of a quiet device."""
    a, c = _inputs(1, 262144, 256, torch.float16, device), _inputs(9, 16384, 320, torch.bfloat16, device)
    want, got, expired = _beside(lambda: torch.cuda._sleep(50_000_000), *a, *c)
    assert expired == 0
    for s, t in zip(got, want):
        for u, v in zip(s, t):
            assert torch.equal(u, v)


def test_beside_kernels_that_fill_the_device(device):
    """The same beside matrix products of another stream, whose workgroups take whole CUs: whether waits expire is then a
    matter of timing, the results are not (statistics that were recomputed are rounded once, from double precision)."""
    a, c = _inputs(1, 262144, 256, torch.float16, device), _inputs(9, 16384, 320, torch.bfloat16, device)
    m = torch.randn(8192, 8192, device=device).bfloat16()
    out = torch.empty_like(m)
    torch.mm(m, m, out=out)
    want, got, expired = _beside(lambda: [torch.mm(m, m, out=out) for _ in range(4)], *a, *c)
    print("expired", expired, flush=True)
    for (y, mean, rstd), (y0, mean0, rstd0) in zip(got, want):
        _close(y, y0, mean, mean0, rstd, rstd0)


def test_cooperative_switch_keeps_to_grids_the_runtime_admits(device):
    """GNNHWC_COOPERATIVE=1 sends single-launch kernels through the runtime's cooperative launch, which refuses a grid larger
    than the device: calls too large to be resident as a whole run on the streaming kernels then, the others as before."""
    import os
    import subprocess
    import sys

    code = """
import sys, torch
from gnnhwc import _cabi
from tests.gpu_harness import cabi_fwd
for N in (2, 9):
    x = torch.randn(N, 16384, 320, device="cuda", dtype=torch.bfloat16)
    w = torch.ones(320, device="cuda", dtype=torch.bfloat16)
    cabi_fwd(x, w, w, 32, 1e-5, 2)
    torch.cuda.synchronize()
    print(_cabi.last_launch().split()[0])
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, GNNHWC_COOPERATIVE="1", PYTHONPATH=os.pathsep.join((root, os.path.join(root, "channels-last-groupnorm_amd"))))
    run = subprocess.run([sys.executable, "-c", code], env=env, cwd=root, capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stderr
    assert run.stdout.split() == ["fused_fwd", "multi-launch"]
