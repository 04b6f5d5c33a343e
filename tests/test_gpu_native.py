"""The native eager route (gnnhwc._native.group_norm, csrc/gn_torch.cpp) against the Python implementation behind the same
public calls: the kernels are the same, so outputs and gradients are equal bit for bit, in every form that the route takes;
and what it does not take it declines, so that those calls and their errors stay the Python implementation's."""
import pytest
import torch

from gnnhwc import GN_NHWC, _native, custom_gn
from gnnhwc.custom_gn import group_norm_nhwc


class Counter:
    """Stands in for the extension inside custom_gn: counts the calls that took the native route, or refuses them all."""

    def __init__(self, refuse=False):
        self.refuse, self.taken = refuse, 0

    def group_norm(self, *args):
        out = NotImplemented if self.refuse else _native.group_norm(*args)
        self.taken += out is not NotImplemented
        return out


def _routes(monkeypatch, fn):
    """fn()'s results by the native route and by the Python one, and how many calls went native."""
    native, python = Counter(), Counter(refuse=True)
    monkeypatch.setattr(custom_gn, "_native", native)
    a = fn()
    monkeypatch.setattr(custom_gn, "_native", python)
    b = fn()
    return a, b, native.taken


def _same(a, b):
    assert len(a) == len(b)
    for s, t in zip(a, b):
        assert (s is None) == (t is None)
        if s is not None:
            assert s.dtype == t.dtype and s.shape == t.shape
            assert [k for k, n in zip(s.stride(), s.shape) if n != 1] == [k for k, n in zip(t.stride(), t.shape) if n != 1]
            assert torch.equal(s, t)


def _channels_last(t):
    nd = t.dim()
    return t.permute(0, *range(2, nd), 1).contiguous().permute(0, nd - 1, *range(1, nd - 1))


@pytest.mark.gpu
@pytest.mark.parametrize("shape,G", [((2, 8, 5), 2), ((1, 64, 7, 9), 8), ((3, 35, 4, 6), 5), ((2, 16, 3, 4, 5), 4), ((2, 8, 1, 1), 2),
                                     ((1, 1, 6, 5), 1)])
@pytest.mark.parametrize("dtype,params", [(torch.float32, torch.float32), (torch.float64, torch.float64),
                                          (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)])
@pytest.mark.parametrize("first", [False, True])
@pytest.mark.parametrize("affine", [True, False])
def test_module_forward_and_backward(shape, G, dtype, params, first, affine, device, monkeypatch):
    torch.manual_seed(1)
    base = torch.randn(shape, device=device).to(dtype)
    base = base if first else _channels_last(base)
    m = GN_NHWC(G, shape[1], activation="silu", affine=affine).to(device).to(params)
    dys = [torch.randn(shape, device=device).to(dtype), _channels_last(torch.randn(shape, device=device).to(dtype)),
           torch.ones((), device=device, dtype=dtype).expand(shape)]

    def fn():
        out = []
        for dy in dys:  # contiguous, channels-last and expanded gradients
            x = base.clone(memory_format=torch.preserve_format).requires_grad_()
            y = m(x)
            out += [y.detach(), *torch.autograd.grad(y, (x, *m.parameters()), dy)]
        with torch.no_grad():
            out.append(m(base))
        return out

    a, b, taken = _routes(monkeypatch, fn)
    _same(a, b)
    assert taken == 4


@pytest.mark.gpu
def test_irregular_strides_and_empty_input_are_declined(device, monkeypatch):
    m = GN_NHWC(2, 8).to(device)
    odd = torch.randn(2, 5, 3, 8, device=device).permute(0, 3, 2, 1)  # channels fastest, spatial dimensions swapped
    cut = torch.randn(2, 16, 5, 3, device=device)[:, :8]              # channels-first, samples not adjacent
    for x in (odd, cut, torch.empty(0, 8, 4, 4, device=device)):
        a, b, taken = _routes(monkeypatch, lambda: [m(x).detach()])
        _same(a, b)
        assert taken == 0


@pytest.mark.gpu
@pytest.mark.parametrize("out", [torch.float16, torch.bfloat16])
def test_cast_output(out, device, monkeypatch):
    m = GN_NHWC(4, 32, activation="gelu", out_dtype=out).to(device)
    base, dy = _channels_last(torch.randn(2, 32, 6, 5, device=device)), torch.randn(2, 32, 6, 5, device=device).to(out)

    def fn():
        x = base.clone(memory_format=torch.preserve_format).requires_grad_()
        y = m(x)
        return [y.detach(), *torch.autograd.grad(y, (x, m.weight, m.bias), dy)]

    a, b, taken = _routes(monkeypatch, fn)
    _same(a, b)
    assert taken == 1


@pytest.mark.gpu
@pytest.mark.parametrize("residual,bias,want", [(True, True, True), (True, False, False), (False, True, True), (False, False, True)])
@pytest.mark.parametrize("cb_type", [torch.bfloat16, torch.float32])
def test_fused_additions(residual, bias, want, cb_type, device, monkeypatch):
    torch.manual_seed(2)
    x, r = (_channels_last(torch.randn(2, 32, 6, 5, device=device).bfloat16()) for _ in range(2))
    cb = torch.randn(2, 32, device=device).to(cb_type)
    w, b = torch.rand(32, device=device).bfloat16(), torch.randn(32, device=device).bfloat16()

    def fn():
        out = group_norm_nhwc(x, w, b, 4, 1e-5, "silu", residual=r if residual else None, channel_bias=cb if bias else None,
                              return_sum=want)
        return list(out) if want else [out]

    a, c, taken = _routes(monkeypatch, fn)
    _same(a, c)
    assert taken == 1
    # with gradients the operators' own autograd formula is the general one
    w2 = w.clone().requires_grad_()
    _, _, taken = _routes(monkeypatch, lambda: group_norm_nhwc(x, w2, b, 4, 1e-5, "silu", residual=r))
    assert taken == 0


@pytest.mark.gpu
def test_saved_tensor_hooks_and_checkpoint_see_the_saved_tensors(device):
    m = GN_NHWC(4, 32, activation="silu").to(device)
    x = _channels_last(torch.randn(2, 32, 6, 5, device=device)).requires_grad_()
    want = torch.autograd.grad(m(x).sum(), (x, m.weight, m.bias))
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t) or t.cpu(), lambda t: t.to(device)):
        y = m(x)
    got = torch.autograd.grad(y.sum(), (x, m.weight, m.bias))
    assert len(seen) >= 4
    for s, t in zip(got, want):
        assert torch.equal(s, t)
    from torch.utils.checkpoint import checkpoint

    got = torch.autograd.grad(checkpoint(m, x, use_reentrant=False).sum(), (x, m.weight, m.bias))
    for s, t in zip(got, want):
        assert torch.equal(s, t)
    # an input changed in place between the passes is still noticed
    z = (x * 1).contiguous(memory_format=torch.channels_last)
    y = m(z)
    z.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


@pytest.mark.gpu
def test_transforms_modes_and_subclasses_are_declined(device, monkeypatch):
    import torch.autograd.forward_ad as fwAD
    from torch.utils._python_dispatch import TorchDispatchMode

    m = GN_NHWC(4, 32).to(device)
    x = _channels_last(torch.randn(2, 32, 6, 5, device=device))
    counter = Counter()
    monkeypatch.setattr(custom_gn, "_native", counter)

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    with Mode():
        m(x)
    m(x.as_subclass(Sub))
    with torch.overrides.BaseTorchFunctionMode():
        m(x)
    with fwAD.dual_level():
        with pytest.raises(Exception):
            m(fwAD.make_dual(x, torch.ones_like(x)))
    with pytest.raises(Exception):
        torch.vmap(m)(x.unsqueeze(0))
    assert counter.taken == 0
    m(x)
    with torch.autocast("cuda", dtype=torch.bfloat16), torch.inference_mode():
        m(x)
    assert counter.taken == 2


@pytest.mark.gpu
def test_streams_threads_and_replayed_graphs(device):
    import threading

    m = GN_NHWC(8, 64, activation="silu").to(device)
    xs = [_channels_last(torch.randn(2, 64, 16, 16, device=device)) for _ in range(4)]
    want = []
    for x in xs:
        x.requires_grad_()
        y = m(x)
        want.append((y.detach(), torch.autograd.grad(y, x, x.detach())[0]))
    got, streams = [None] * 4, [torch.cuda.Stream() for _ in range(4)]
    torch.cuda.synchronize()

    def work(i):
        with torch.cuda.stream(streams[i]):
            for _ in range(10):
                y = m(xs[i])
                got[i] = (y.detach(), torch.autograd.grad(y, xs[i], xs[i].detach())[0])

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert torch.equal(g[0], w[0]) and torch.equal(g[1], w[1])
    graph, static = torch.cuda.CUDAGraph(), xs[0].detach().clone(memory_format=torch.preserve_format)
    with torch.no_grad():
        m(static)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            out = m(static)
        for x, w in zip(xs, want):
            static.copy_(x.detach())
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, w[0])
            m(x)


def test_host_tensors_are_declined():
    x = torch.randn(2, 8, 4, 4)
    w, b = torch.ones(8), torch.zeros(8)
    assert _native.group_norm(x, w, b, 2, 1e-5, 0, None, None, None, False) is NotImplemented
    assert _native.group_norm(None, w, b, 2, 1e-5, 0, None, None, None, False) is NotImplemented
    with pytest.raises(RuntimeError):
        _native.group_norm(x)


# What unpacking hooks may hand to the backward in place of the saved tensors, each with equal values: other strides (what
# offloading hooks that pack into empty(size) return), a view into a larger buffer, a broadcastable stride pattern undone.
def _contiguous(t):
    return t.contiguous(memory_format=torch.contiguous_format).clone(memory_format=torch.contiguous_format)


def _cut(t):
    buf = t.new_empty((2, *t.shape))
    buf[1] = t
    return buf[1]


def _reversed_dims(t):
    return t.permute(*reversed(range(t.dim()))).contiguous().permute(*reversed(range(t.dim())))


@pytest.mark.gpu
@pytest.mark.parametrize("unpack", [_contiguous, _cut, _reversed_dims])
@pytest.mark.parametrize("functional", [False, True])
@pytest.mark.parametrize("shape,first", [((2, 32, 6, 5), False), ((2, 32, 6, 5), True), ((3, 8, 3, 4, 5), False), ((2, 12, 7), False)])
def test_saved_tensors_may_come_back_in_any_layout(unpack, functional, shape, first, device):
    if functional and first:
        pytest.skip("group_norm_nhwc takes channels-last input only")
    m = GN_NHWC(4, shape[1], activation="silu").to(device)
    x = torch.randn(shape, device=device)
    x = (x if first else _channels_last(x)).requires_grad_()
    dy = torch.randn(shape, device=device)
    call = (lambda: group_norm_nhwc(x, m.weight, m.bias, 4, m.eps, "silu")) if functional else (lambda: m(x))
    want = torch.autograd.grad(call(), (x, m.weight, m.bias), dy)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        y = call()
    for s, t in zip(torch.autograd.grad(y, (x, m.weight, m.bias), dy), want):
        assert torch.equal(s, t)


@pytest.mark.gpu
@pytest.mark.parametrize("pin", [False, True])
def test_save_on_cpu(pin, device):
    m = GN_NHWC(4, 32, activation="gelu").to(device)
    x, dy = (_channels_last(torch.randn(2, 32, 6, 5, device=device)) for _ in range(2))
    x.requires_grad_()
    want = torch.autograd.grad(m(x), (x, m.weight, m.bias), dy)
    with torch.autograd.graph.save_on_cpu(pin_memory=pin):
        y = m(x)
    for s, t in zip(torch.autograd.grad(y, (x, m.weight, m.bias), dy), want):
        assert torch.equal(s, t)


@pytest.mark.gpu
def test_saved_tensors_of_another_device_type_or_size_are_refused(device):
    m = GN_NHWC(4, 32).to(device)
    x = _channels_last(torch.randn(2, 32, 6, 5, device=device)).requires_grad_()
    for pick, change, message in [(4, lambda t: t.cpu(), "must be a CUDA tensor"), (1, lambda t: t.cpu(), "must be a CUDA tensor"),
                                  (3, lambda t: t.cpu(), "must be a CUDA tensor"), (4, lambda t: t.half(), "same dtype"),
                                  (1, lambda t: t[:16], "32 elements"), (4, lambda t: t[:1], "same shape"), (3, lambda t: t[:1], "N\\*G")]:
        # pick: the parameters (1 dimension), the statistics (3) or x (4)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: change(t) if t.dim() == pick else t):
            y = m(x)
        with pytest.raises(RuntimeError, match=message):
            y.sum().backward()


# Backwards that are no ordinary call go through the operators, whose formula group_norm_nhwc's derivative is.
@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:There is a performance drop")
@pytest.mark.parametrize("out", [None, torch.bfloat16])
@pytest.mark.parametrize("shape", [(2, 32, 6, 5), (2, 12, 7), (1, 8, 3, 4, 5)])
def test_batched_gradients_of_the_functional_form(shape, out, device):
    m = GN_NHWC(4, shape[1]).to(device)
    x = _channels_last(torch.randn(shape, device=device)).requires_grad_()
    y = group_norm_nhwc(x, m.weight, m.bias, 4, m.eps, "silu", out_dtype=out)
    dys = torch.randn((3, *shape), device=device).to(y.dtype)
    got = torch.autograd.grad(y, (x, m.weight, m.bias), dys, retain_graph=True, is_grads_batched=True)
    for i in range(3):
        want = torch.autograd.grad(y, (x, m.weight, m.bias), dys[i], retain_graph=True)
        for s, t in zip(got, want):
            assert torch.equal(s[i], t)
    small = _channels_last(torch.randn(1, 4, 2, device=device))
    jac = torch.autograd.functional.jacobian(lambda t: group_norm_nhwc(t, m.weight[:4].detach(), m.bias[:4].detach(), 2), small, vectorize=True)
    want = torch.autograd.functional.jacobian(lambda t: torch.nn.functional.group_norm(t, 2, m.weight[:4], m.bias[:4]), small)
    assert (jac - want).abs().max() <= 1e-5 * want.abs().max()


@pytest.mark.gpu
def test_the_functional_forms_backward_is_seen_by_modes_and_graphs(device):
    from torch.utils._python_dispatch import TorchDispatchMode

    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    m = GN_NHWC(4, 32, activation="silu").to(device)
    x = _channels_last(torch.randn(2, 32, 6, 5, device=device)).requires_grad_()
    y = group_norm_nhwc(x, m.weight, m.bias, 4, m.eps, "silu")
    want = torch.autograd.grad(y, (x, m.weight, m.bias), x.detach(), retain_graph=True)
    with Mode():
        got = torch.autograd.grad(y, (x, m.weight, m.bias), x.detach(), retain_graph=True)
    assert "gnop.bwd.default" in seen
    again = torch.autograd.grad(y, (x, m.weight, m.bias), x.detach(), create_graph=True)
    for s, t, u in zip(got, want, again):
        assert torch.equal(s, t) and torch.equal(u, t)
        assert u.requires_grad  # the operator has no second derivative: autograd's fallback notes it and warns when it is asked for
    # the module's own function never recorded its backward
    assert not any(g.requires_grad for g in torch.autograd.grad(m(x), (x, m.weight, m.bias), x.detach(), create_graph=True))


@pytest.mark.gpu
def test_gradients_of_another_kind_through_the_module(device):
    class Sub(torch.Tensor):
        pass

    for first in (False, True):
        m = GN_NHWC(4, 32, activation="silu").to(device)
        x = torch.randn(2, 32, 6, 5, device=device)
        x = (x if first else _channels_last(x)).requires_grad_()
        dys = torch.randn(3, 2, 32, 6, 5, device=device)
        y = m(x)
        want = [torch.autograd.grad(y, (x, m.weight, m.bias), d, retain_graph=True) for d in dys]
        got = torch.autograd.grad(y, (x, m.weight, m.bias), dys, retain_graph=True, is_grads_batched=True)
        for i in range(3):
            for s, t in zip(got, want[i]):
                assert torch.equal(s[i], t)
        for s, t in zip(torch.autograd.grad(y, (x, m.weight, m.bias), dys[0].as_subclass(Sub)), want[0]):
            assert torch.equal(s, t)
    bare = GN_NHWC(4, 32, affine=False).to(device)
    y = bare(x)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(y, x, dys, is_grads_batched=True)


@pytest.mark.gpu
@pytest.mark.parametrize("first", [False, True])
def test_the_interpreter_lock_is_released_around_the_kernels(first, device):
    """The extension's launches are replaced by CPython's own question whether the calling thread holds the lock: an answer
    other than 0 is an error code of the launch."""
    import ctypes

    from gnnhwc import _cabi

    asked = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    real = [ctypes.cast(getattr(_cabi.lib, "gnnhwc_" + name), ctypes.c_void_p).value for name in _cabi.NATIVE_ENTRY_POINTS]
    launches = ("fwd_cast", "bwd_cast", "fwd_add", "fwd_nchw", "bwd_nchw")
    m = GN_NHWC(4, 32).to(device)
    x = torch.randn(2, 32, 6, 5, device=device)
    x = x if first else _channels_last(x)
    dy = torch.zeros_like(x)
    _native.bind(*[asked if name in launches else address for name, address in zip(_cabi.NATIVE_ENTRY_POINTS, real)])
    try:
        with torch.no_grad():
            m(x)
            if not first:
                group_norm_nhwc(x, m.weight, m.bias, 4, residual=x, return_sum=True)
        x.requires_grad_()
        torch.autograd.grad(m(x), x, dy)
    finally:
        _native.bind(*real)
    torch.cuda.synchronize()


@pytest.mark.gpu
def test_calls_appear_under_their_operators_names_in_the_profiler(device):
    from torch.profiler import ProfilerActivity, profile

    m = GN_NHWC(4, 32, activation="silu").to(device)
    x = torch.randn(2, 32, 6, 5, device=device)
    last = _channels_last(x).requires_grad_()
    first = x.clone().requires_grad_()
    with profile(activities=[ProfilerActivity.CPU]) as p:
        m(last).sum().backward()
        m(first).sum().backward()
        with torch.no_grad():
            group_norm_nhwc(last, m.weight, m.bias, 4, residual=last)
            GN_NHWC(4, 32, out_dtype=torch.bfloat16).to(device)(last)
    names = [e.key for e in p.key_averages()]
    for name in ("gnop::fwd", "gnop::bwd", "gnop::fwd_nchw", "gnop::bwd_nchw", "gnop::fwd_add", "gnop::fwd_cast"):
        assert name in names, (name, names)


@pytest.mark.gpu
@pytest.mark.parametrize("affine", [True, False])
@pytest.mark.parametrize("out", [None, torch.bfloat16])
def test_gradients_with_a_tangent(affine, out, device):
    """The operators have no forward-mode derivative: a tangent of the gradient is dropped, the gradients are the same."""
    import torch.autograd.forward_ad as fwAD

    m = GN_NHWC(4, 32, activation="silu", affine=affine, out_dtype=out).to(device)
    x = _channels_last(torch.randn(2, 32, 6, 5, device=device)).requires_grad_()
    dy = torch.randn(2, 32, 6, 5, device=device).to(out or torch.float32)
    inputs = (x, *m.parameters())
    y = m(x)
    want = torch.autograd.grad(y, inputs, dy, retain_graph=True)
    with fwAD.dual_level():
        got = torch.autograd.grad(y, inputs, fwAD.make_dual(dy, torch.ones_like(dy)))
        got = [fwAD.unpack_dual(t).primal.clone() for t in got]
    for s, t in zip(got, want):
        assert torch.equal(s, t)


@pytest.mark.gpu
@pytest.mark.parametrize("first,dtype,out", [(False, torch.bfloat16, None), (False, torch.float32, torch.float16),
                                             (False, torch.float64, None), (True, torch.float16, None), (True, torch.float32, None)])
@pytest.mark.parametrize("shape,G", [((2, 64, 8, 8), 8), ((3, 35, 9, 13), 5), ((1, 128, 600, 500), 32)])
def test_result_without_a_graph_equals_the_one_with(first, dtype, out, shape, G, device):
    """Without a graph the kernels are given nowhere to leave the statistics."""
    torch.manual_seed(2)
    x = torch.randn(shape, device=device).to(dtype)
    x = x if first else _channels_last(x)
    m = GN_NHWC(G, shape[1], activation="gelu", out_dtype=out).to(device).to(dtype)
    with torch.no_grad():
        y = m(x)
    want = m(x.clone().requires_grad_())
    assert want.grad_fn is not None and y.grad_fn is None
    _same((y,), (want.detach(),))
