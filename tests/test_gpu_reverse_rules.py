"""The plain reverse-mode route (autograd functions that hand out the values alone and save
their factors) against the torch.func route of the same calls, over every dtype and the
kernel families it dispatches between: the gradient, a second backward of a retained graph,
saved-tensor hooks, calls under no_grad, and a trace that is replayed on other inputs."""

import numpy as np
import pytest
import torch

import fermix_amd

pytestmark = pytest.mark.gpu

CASES = [(op, n, dt) for op in ("slogdet", "slogpf", "det", "pf") for n, dt in (
    (12, torch.float32), (40, torch.float32), (136, torch.float32),
    (12, torch.float64), (40, torch.float64), (24, torch.complex64), (40, torch.complex128))]


def _make(dev, op, n, dt):
    g = torch.Generator(device=dev).manual_seed(31 * n)
    A = 0.25 * torch.randn(4, n, n, generator=g, device=dev, dtype=dt) / n**0.5
    J = torch.zeros(n, n, device=dev, dtype=dt)
    if op in ("slogpf", "pf"):
        i = torch.arange(0, n, 2, device=dev)
        J[i, i + 1], J[i + 1, i] = 1, -1
    else:
        J += torch.eye(n, device=dev, dtype=dt)
    return A + J


def _value(out):
    return out[1] if isinstance(out, tuple) else out


@pytest.mark.parametrize("op,n,dt", CASES)
def test_reverse_rules(dev, op, n, dt):
    f = getattr(fermix_amd, op)
    A = _make(dev, op, n, dt)
    print(f"reverse rules {op} n={n} {dt}", flush=True)
    w = torch.linspace(0.5, 1.5, 4, device=dev, dtype=_value(f(A)).dtype)
    X = A.clone().requires_grad_()
    v = _value(f(X))
    assert torch.equal(v, _value(f(A))) and v.requires_grad
    (g1,) = torch.autograd.grad(v, X, w, retain_graph=True)
    (g2,) = torch.autograd.grad(v, X, w)
    assert torch.equal(g1, g2)
    _, pull = torch.func.vjp(lambda a: _value(f(a)), A)
    (gf,) = pull(w)
    # the torch.func route scales the finished inverse: a rounding or two apart
    eps = torch.finfo(dt).eps
    assert torch.linalg.vector_norm(g1 - gf) <= 8 * n * eps * torch.linalg.vector_norm(gf)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(dev)):
        v = _value(f(X))
    (g3,) = torch.autograd.grad(v, X, w)
    assert torch.equal(g1, g3)
    with torch.no_grad():
        out = f(X)
    assert not _value(out).requires_grad and torch.equal(_value(out), _value(f(A)))


def test_trace_replays_on_other_inputs(dev):
    """A traced call records the computation, not the first input's values."""
    A, B = _make(dev, "slogdet", 40, torch.float32), 2 * _make(dev, "slogdet", 40, torch.float32)
    t = torch.jit.trace(lambda a: fermix_amd.slogdet(a)[1], (A,), check_trace=False)
    assert np.array_equal(t(B).cpu().numpy(), fermix_amd.slogdet(B)[1].cpu().numpy())
