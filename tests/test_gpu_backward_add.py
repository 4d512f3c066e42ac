"""The stream gradient of the post phase added inside the pre phase's backward
launch: bit for bit what autograd's separate addition gives, on every kernel that
takes it, at the edges of their tiles; and the calls that get no such gradient."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from model import _hip as H  # noqa: E402
from model import _ops  # noqa: E402
from model.mhc_fused import MHCConnection_Fused, _PostPhaseFullFn, _PreSinkhornFn  # noqa: E402
from model.mhc_fused_no_hres import MHCConnection_FusedNoHres, _PostPhaseFn, _PrePhaseFn  # noqa: E402

F32, BF, F16 = torch.float32, torch.bfloat16, torch.float16


def _module(kind, n, C, dt, dev):
    torch.manual_seed(n * C)
    m = (MHCConnection_Fused if kind == "full" else MHCConnection_FusedNoHres)(n, C)
    with torch.no_grad():
        for name, p in m.named_parameters():
            if name.startswith("alpha"):
                p.fill_(0.5)
            elif name.startswith("bias"):
                p.add_(torch.randn(p.shape) * 0.3)
    return m.to(dev).to(dt)


def _apart(m, x, f):
    """The connection with its two uses of x summed by autograd."""
    if isinstance(m, MHCConnection_Fused):
        z, h_post, h_res = _PreSinkhornFn.apply(
            x, m.phi_weight, _ops.packed_phi(m.phi_weight, m.n, m.dim, H.MODE_FULL, True),
            m.alpha_pre, m.bias_pre, m.alpha_post, m.bias_post, m.alpha_res, m.bias_res, 2.0, 1e-6,
            1e-6, m.n, m.dim, m.sinkhorn_iters, 1e-6)
        return _PostPhaseFullFn.apply(x, h_res, h_post, f(z), m.n, m.dim)
    z, _, h_post = _PrePhaseFn.apply(x, m.phi_weight, m.alpha_pre, m.bias_pre, m.alpha_post,
                                     m.bias_post, 2.0, 1e-6, 1e-6, m.n, m.dim)
    return _PostPhaseFn.apply(x, h_post, f(z), m.n, m.dim)


def _grads(m, out, x, g):
    return torch.autograd.grad(out, [x, *m.parameters()], g, retain_graph=True)


@pytest.mark.parametrize("kind,n,C,dt,shape", [
    ("full", 4, 768, BF, (1, 1)), ("full", 4, 768, BF, (3, 37)), ("full", 4, 768, F32, (2, 33)),
    ("full", 8, 512, BF, (1, 47)), ("full", 8, 768, F32, (1, 17)), ("full", 2, 64, BF, (1, 16)),
    ("full", 4, 200, BF, (1, 31)), ("full", 4, 200, F32, (1, 15)), ("full", 4, 1024, F32, (1, 50)),
    ("full", 16, 64, BF, (1, 9)), ("full", 4, 96, F16, (1, 21)), ("full", 4, 1536, BF, (1, 5)),
    ("nohres", 4, 768, BF, (2, 70)), ("nohres", 8, 72, BF, (1, 33)), ("nohres", 4, 256, F32, (1, 18)),
    ("nohres", 2, 40, BF, (1, 3))])
def test_same_bits_as_a_separate_addition(dev, kind, n, C, dt, shape):
    m = _module(kind, n, C, dt, dev)
    x = torch.randn(*shape, n * C, device=dev).to(dt).requires_grad_()
    g = torch.randn(*shape, n * C, device=dev).to(dt)
    low = (lambda z: z.to(BF)) if dt == F32 else (lambda z: z * 1.5)
    out, ref = m(x, low), _apart(m, x, low)
    assert torch.equal(out, ref)
    for got, want in zip(_grads(m, out, x, g), _grads(m, ref, x, g)):
        assert torch.equal(got, want)


def test_strided_and_expanded_gradients(dev):
    m = _module("full", 4, 64, BF, dev)
    x = torch.randn(2, 5, 256, device=dev).to(BF).requires_grad_()
    for g in (torch.randn(5, 2, 256, device=dev).to(BF).transpose(0, 1),
              torch.ones(1, 1, 1, device=dev).to(BF).expand(2, 5, 256)):
        got, = torch.autograd.grad(m(x, torch.tanh), x, g)
        want, = torch.autograd.grad(_apart(m, x, torch.tanh), x, g)
        assert torch.equal(got, want)


@pytest.mark.parametrize("kind", ["full", "nohres"])
def test_partial_graphs(dev, kind):
    """A stream without a gradient, a sublayer that ignores its input, an output
    that is only the sublayer's, and frozen parameters."""
    m = _module(kind, 4, 64, BF, dev)
    x = torch.randn(1, 6, 256, device=dev).to(BF)
    f = torch.randn(1, 6, 64, device=dev).to(BF)
    g = torch.randn(1, 6, 256, device=dev).to(BF)
    for sub in (torch.tanh, lambda z: f):
        got = torch.autograd.grad(m(x, sub), list(m.parameters()), g, allow_unused=True)
        want = torch.autograd.grad(_apart(m, x, sub), list(m.parameters()), g, allow_unused=True)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    seen = []
    xr = x.clone().requires_grad_()
    m(xr, lambda z: seen.append(z) or z)
    got, = torch.autograd.grad(seen[0].float().sum(), xr)  # nothing through the post phase
    assert torch.isfinite(got).all() and float(got.abs().max()) > 0
    m.requires_grad_(False)
    got, = torch.autograd.grad(m(xr, torch.tanh), xr, g)
    want, = torch.autograd.grad(_apart(m, xr, torch.tanh), xr, g)
    assert torch.equal(got, want)


def test_hooks_and_saved_tensor_hooks(dev):
    m = _module("full", 4, 64, BF, dev)
    x = torch.randn(1, 6, 256, device=dev).to(BF).requires_grad_()
    y = x * 1.0
    seen = []
    y.register_hook(lambda g: seen.append(g.clone()))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(dev)):
        out = m(y, torch.tanh)
    out.float().sum().backward()
    assert len(seen) == 1 and torch.equal(seen[0], x.grad)
    want, = torch.autograd.grad(_apart(m, x, torch.tanh).float().sum(), x)
    assert torch.equal(x.grad, want)


@pytest.mark.parametrize("kind", ["full", "nohres"])
def test_no_sum_for_a_stream_without_a_gradient(dev, kind, monkeypatch):
    """A stream that needs no gradient has none to add: the launch reads one stream less."""
    m = _module(kind, 4, 64, BF, dev)
    x = torch.randn(1, 6, 256, device=dev).to(BF)
    added, pre_bwd = [], _ops.pre_bwd

    def spy(*args, g_x_in=None, **kwargs):
        added.append(g_x_in is not None)
        return pre_bwd(*args, g_x_in=g_x_in, **kwargs)

    monkeypatch.setattr(_ops, "pre_bwd", spy)
    for xx in (x, x.clone().requires_grad_()):
        m(xx, torch.tanh).float().sum().backward()
    assert added == [False, True]


@pytest.mark.parametrize("kind,n,C,dt", [("nohres", 4, 64, BF), ("nohres", 2, 96, F32), ("full", 4, 64, BF)])
def test_gradient_off_16_byte_alignment(dev, kind, n, C, dt):
    """A gradient that arrives at an odd offset (without a residual matrix it is the one
    that the pre phase adds, as it came) leaves the pre phase on its MFMA kernel."""
    m = _module(kind, n, C, dt, dev)
    x = torch.randn(2, 9, n * C, device=dev).to(dt).requires_grad_()
    buf = torch.randn(x.numel() + 1, device=dev).to(dt)
    g = buf[1:].view(x.shape)
    assert g.data_ptr() % 16 and g.is_contiguous()
    low = (lambda z: z.to(BF)) if dt == F32 else torch.tanh
    for got, want in zip(_grads(m, m(x, low), x, g), _grads(m, _apart(m, x, low), x, g)):
        assert torch.equal(got, want)
