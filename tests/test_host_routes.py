"""Which native call a public entry point makes, and what it refuses, with the launches
replaced: no GPU needed."""
import ctypes

import pytest
import torch
import torch.nn as nn

from tbf16 import _ext
from tbf16 import conv as tconv


def _converted(C, O, k=3, **kw):
    """A converted Conv2d on the CPU (convert_conv without its quantisation kernel)."""
    m = nn.Conv2d(C, O, k, **kw).bfloat16()
    w16 = m.weight.detach().half()
    m.weight = None
    m.register_buffer("weight16", w16)
    m.register_buffer("weight_scale", torch.ones(O))
    m._tbf16_plan = tconv.ConvPlan(0, tconv._pointwise(m))
    m.__class__ = tconv._scaled_class(type(m))
    return m


@pytest.fixture
def conv_calls(monkeypatch):
    """The native calls that a converted convolution on CPU tensors would launch."""
    calls = []
    monkeypatch.setattr(tconv, "_dev_check", lambda *ts: None)
    monkeypatch.setattr(tconv, "launch", lambda name, *args: calls.append(name))
    monkeypatch.setattr(tconv, "scale_input", lambda x, t: (torch.zeros(x.shape[0], dtype=torch.int32), x.half()))
    monkeypatch.setattr(tconv, "unscale_output", lambda y16, *args: y16.bfloat16())
    return calls


@pytest.mark.parametrize("C", [256, 1024, 4])
@pytest.mark.parametrize("cl", [False, True])
def test_conv2d_of_other_channel_counts_is_refused(conv_calls, C, cl):
    m = _converted(512, 512, padding=1)
    fmt = torch.channels_last if cl else torch.contiguous_format
    with torch.no_grad():
        m(torch.zeros(1, 512, 64, 64, dtype=torch.bfloat16).to(memory_format=fmt))
        assert conv_calls == ["tbf16_conv2d"]
        with pytest.raises(RuntimeError, match="channels"):  # torch's own error
            m(torch.zeros(1, C, 64, 64, dtype=torch.bfloat16).to(memory_format=fmt))
    assert conv_calls == ["tbf16_conv2d"]


def test_conv2d_entry_point_refuses_other_channel_counts():
    two = (ctypes.c_int64 * 2)(1, 1)
    for C in (256, 1024):
        rc = _ext.lib().tbf16_conv2d(16, 1, C, 64, 64, 0, 0, 16, 512, 512, 3, 3, two, two, two, 16, None, 16, 16, 1 << 40, None)
        assert rc == -1 and "channels" in _ext.lib().tbf16_last_error().decode()


@pytest.fixture
def linear_calls(monkeypatch):
    """The native calls of the training linear on CPU tensors, as (name, arguments)."""
    from tbf16 import autograd, ops, routing
    calls = []
    monkeypatch.setattr(ops, "_dev_check", lambda *ts: None)
    for mod in (ops, autograd):
        monkeypatch.setattr(mod, "launch", lambda name, where, *args: calls.append((name, args)))
    routing.activations.clear()
    yield calls
    routing.activations.clear()


@pytest.mark.parametrize("N", [12, 1025])
def test_linear_input_gradient_of_any_n(linear_calls, N):
    """dX = dY W of a frozen layer whose N is no multiple of 8: the product's two operands
    have one (padded) contraction length."""
    from tbf16 import autograd
    x = torch.zeros(10, 16, dtype=torch.bfloat16, requires_grad=True)
    y = autograd.linear(x, torch.zeros(N, 16, dtype=torch.bfloat16))
    assert y.shape == (10, N)
    (dx,) = torch.autograd.grad(y, [x], torch.zeros(10, N, dtype=torch.bfloat16))
    assert dx.shape == (10, 16)
    name, args = linear_calls[-1]
    assert name == "tbf16_gemm_f16" and args[1:4] == (10, N + -N % 8, N + -N % 8)


@pytest.mark.parametrize("N", [12, 1025])
def test_linear_of_any_n_takes_a_misaligned_weight(linear_calls, N):
    """A weight that does not start on 16 bytes (a view into a packed buffer) is copied for the
    kernels, whose entry points refuse it."""
    from tbf16 import ops
    w16 = torch.zeros(N * 16 + 1, dtype=torch.float16)[1:].view(N, 16)
    assert w16.data_ptr() % 16
    x16 = torch.zeros(40, 16, dtype=torch.float16)
    y = ops.linear_q(x16, torch.ones(40), w16, torch.ones(N))
    (name, args), = linear_calls
    assert y.shape == (40, N) and name == "tbf16_gemm_f16_any_n" and args[5] not in (0, None) and args[5] % 16 == 0


@pytest.mark.parametrize("K,N", [(16, 12), (30, 40), (13, 1025)])
def test_linear_gradients_have_their_leaves_shapes(linear_calls, K, N):
    from tbf16 import autograd
    leaves = [torch.zeros(*s, dtype=torch.bfloat16, requires_grad=True) for s in ((10, K), (N, K), (N,))]
    y = autograd.linear(*leaves)
    grads = torch.autograd.grad(y, leaves, torch.zeros(10, N, dtype=torch.bfloat16))
    assert [g.shape for g in grads] == [t.shape for t in leaves]


@pytest.mark.parametrize("M,K,N", [(40, 64, 24), (33, 1, 16), (10, 30, 12)])
def test_linear_takes_an_activation_of_any_strides(linear_calls, M, K, N):
    """A transposed activation, or one whose columns are not side by side."""
    from tbf16 import autograd
    for x in (torch.zeros(K, M, dtype=torch.bfloat16).t(), torch.zeros(M, 3 * K, dtype=torch.bfloat16)[:, ::3]):
        x = x.detach().requires_grad_()
        y = autograd.linear(x, torch.zeros(N, K, dtype=torch.bfloat16))
        (dx,) = torch.autograd.grad(y, [x], torch.zeros_like(y))
        assert y.shape == (M, N) and dx.shape == x.shape


def test_linear_refuses_host_tensors(linear_calls, monkeypatch):
    """A weight (or a saved tensor that a hook unpacked) in host memory raises before any
    launch: its address must not reach a kernel."""
    from tbf16 import autograd, ops
    monkeypatch.undo()  # the real device check
    calls = []
    for mod in (ops, autograd):
        monkeypatch.setattr(mod, "launch", lambda name, where, *args: calls.append(name))
    x = torch.zeros(16, 16, dtype=torch.bfloat16, requires_grad=True)
    w = torch.zeros(24, 16, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="device"):
        autograd.linear(x, w)
    assert calls == []
    checked = []
    monkeypatch.setattr(ops, "_dev_check", lambda *ts: checked.append(len(ts)))
    y = autograd.linear(x, w)
    checked.clear()
    torch.autograd.grad(y, [x], torch.zeros_like(y))
    assert checked and calls[-1] == "tbf16_train_linear_bwd"


@pytest.mark.parametrize("unpack", [lambda t: t.t().contiguous().t(), lambda t: torch.cat([t, t], 1)[:, :t.shape[1]]])
def test_linear_backward_takes_saved_tensors_of_any_layout(linear_calls, unpack):
    """Saved-tensor hooks may give x's transposed copy back with other strides: those go pass
    by pass, where operands are made contiguous."""
    from tbf16 import autograd
    x = torch.zeros(16, 32, dtype=torch.bfloat16, requires_grad=True)
    w = torch.zeros(24, 32, dtype=torch.bfloat16, requires_grad=True)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: unpack(t) if t.dtype == torch.float16 else t):
        y = autograd.linear(x, w)
        grads = torch.autograd.grad(y, [x, w], torch.zeros_like(y))
    assert [g.shape for g in grads] == [x.shape, w.shape]
    assert "tbf16_train_linear_bwd" not in [name for name, _ in linear_calls]


@pytest.mark.parametrize("cast", [torch.bfloat16, torch.float32])
def test_conv2d_cast_after_conversion_is_refused(conv_calls, cast):
    """A model cast after its conversion has a weight that is no fp16 any more: torch's own
    error, as its bits must not be read as fp16."""
    m = _converted(128, 128, padding=1).to(cast)
    m.bias = nn.Parameter(m.bias.detach().bfloat16())
    with torch.no_grad(), pytest.raises(RuntimeError):
        m(torch.zeros(1, 128, 64, 64, dtype=torch.bfloat16))
    assert conv_calls == []


def test_conv2d_bias_in_host_memory_is_refused(conv_calls, monkeypatch):
    """The native convolution checks every operand that it reads, the bias too."""
    seen = []
    monkeypatch.setattr(tconv, "_dev_check", lambda *ts: seen.extend(t.data_ptr() for t in ts if t is not None))
    m = _converted(128, 128, padding=1)
    x = torch.zeros(1, 128, 64, 64, dtype=torch.bfloat16)
    with torch.no_grad():
        m(x)
    assert {t.data_ptr() for t in (x, m.weight16, m.weight_scale, m.bias)} <= set(seen)


@pytest.mark.parametrize("N", [24, 12])
def test_linear_keeps_one_copy_of_an_activation(linear_calls, N):
    """What the memo keeps while x lives is the transposed fp16 copy and its scales, which the
    backward saves anyway: a second copy for each of eight activations is memory that a
    model may not have. A second layer on x makes no second transposed copy."""
    from tbf16 import autograd, routing
    M, K = 40, 64
    x = torch.zeros(M, K, dtype=torch.bfloat16, requires_grad=True)
    ws = [torch.zeros(N, K, dtype=torch.bfloat16, requires_grad=True) for _ in range(2)]
    autograd.linear(x, ws[0])
    (_, kept), = routing.activations._entries.values()
    assert sum(t.numel() * t.element_size() for t in kept) <= 2 * K * M + 4 * M
    first = len(linear_calls)
    autograd.linear(x, ws[1])
    (_, again), = routing.activations._entries.values()
    assert all(a is b for a, b in zip(kept, again))
    assert kept[0].data_ptr() not in [a for _, args in linear_calls[first:] for a in args]


@pytest.mark.parametrize("M,N,K", [(8193, 2048, 768), (4096, 32000, 768), (8193, 4096, 64)])
def test_linear_backward_workspace_holds_what_is_wanted(M, N, K):
    """The backward's workspace: W's fp16 columns and dY's rows for dX, dY's columns for dW, and
    where dY is large its two copies in one place; the rest is vectors and three sets of at most 2^21 partial results."""
    ws = lambda *want: _ext.lib().tbf16_train_linear_bwd_ws_bytes(M, N, K, *want)
    W, dY = 2 * N * K, 2 * N * (M + -M % 8)
    rest = 32 * (M + N + K) + 3 * (9 << 20)
    assert W + dY <= ws(1, 0, 0) + 16 * N <= W + dY + rest
    assert dY <= ws(0, 1, 0) <= dY + rest
    assert ws(0, 0, 1) <= rest
    assert W + dY <= ws(1, 1, 1) <= W + dY + rest + (dY if 2 * M * N < 64 << 20 else 0)


@pytest.mark.parametrize("B,C,O,side,k,native", [
    (1, 8, 8, 1024, 3, False), (1, 16, 16, 512, 3, False),     # 8 and 4 times the input's memory
    (1, 3, 64, 512, 5, False), (1, 4, 320, 512, 3, False),     # few channels, large images
    (1, 96, 16, 1024, 3, False), (1, 96, 64, 1024, 3, True),   # 128 channels against 96 + O
    (1, 3, 320, 450, 11, False), (1, 8, 320, 450, 7, False), (1, 16, 320, 400, 5, False),  # products with zeros
    (1, 4, 64, 300, 5, True), (1, 24, 320, 400, 7, True), (1, 32, 320, 400, 5, True),
    (1, 16, 64, 256, 3, True), (2, 16, 64, 224, 7, True), (1, 512, 512, 128, 3, True), (1, 64, 64, 512, 3, True),
])
@pytest.mark.parametrize("cl", [False, True])
def test_conv2d_route_by_the_padded_copy(B, C, O, side, k, native, cl):
    """The native kernels pad the input's channels to a multiple of 64. They are used where
    that copy is small, or no larger than the library path's own fp16 copies, and not too many
    products are with zeros."""
    if cl and C % 8:
        pytest.skip("channels last takes channels in multiples of 8")
    m = _converted(C, O, k, padding=k // 2)
    x = torch.empty(B, C, side, side, dtype=torch.bfloat16, device="meta")
    x = x.to(memory_format=torch.channels_last) if cl else x
    assert tconv._native_layout(m, x, m.padding, m.bias) == (int(cl) if native else None)
