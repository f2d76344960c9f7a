"""Calls whose matrix is closed over inside a torch.func transform of something else (a
parameter of a model that is vmapped over samples): it is no wrapped tensor, yet a
transform is active. The routing of all four functions, with the kernel calls replaced by
torch (no GPU): values, the gradient of the closed-over matrix, and raw pointers of every
tensor that a kernel call would be handed."""

import pytest
import torch

import fermix_amd
from fermix_amd import _diff, _kernels

torch_slogdet = torch.linalg.slogdet


def _pf(S):
    """pf of real even-order skew matrices, by its expansion along the first row."""
    n = S.shape[-1]
    if n == 0:
        return torch.ones(S.shape[:-2], dtype=S.dtype)
    total = 0
    for j in range(1, n):
        keep = [i for i in range(n) if i not in (0, j)]
        total = total + (-1) ** (j - 1) * S[..., 0, j] * _pf(S[..., keep, :][..., :, keep])
    return total


def _skew(A, skew):
    return (A - A.transpose(-1, -2)) / 2 if skew else A


def _raw(*ts):
    for t in ts:
        if t is not None:
            t.data_ptr()  # refused for a transform's wrapper


def _out(x):
    """As a kernel leaves it: a new tensor from torch.empty, written through its pointer."""
    y = torch.empty(x.shape, dtype=x.dtype)
    _raw(y)
    return y.copy_(x)


def _stub(mp):
    def slogdet(A, x3=0):
        _raw(A)
        s, l = torch_slogdet(A.detach())
        return _out(s), _out(l)

    def slogdet_parts(A, x3=0):
        return (*slogdet(A), _out(torch.linalg.inv(A.detach()).transpose(-1, -2)), None, None)

    def slogdet_factors(A, x3=0):
        return (*slogdet(A), _out(A.detach()), torch.zeros(A.shape[:-1], dtype=torch.int32))

    def slogdet_inverse(lu, perm, sign, n, scale=None, x3=0):
        _raw(lu, perm, sign, scale)
        return _out(scale[:, None, None] * torch.linalg.inv(lu).transpose(-1, -2))

    def det_parts(A, x3=0):
        s, l = slogdet(A)
        return s, l, _out((s * l.exp())[:, None, None] * torch.linalg.inv(A.detach()).transpose(-1, -2))

    def slogpf(A, skew, x3=0):
        _raw(A)
        p = _pf(_skew(A.detach(), skew)) if A.shape[-1] <= 8 else torch.linalg.det(_skew(A.detach(), skew)).sqrt()
        return _out(p.sign()), _out(p.abs().log())

    def slogpf_parts(A, skew, adjugate=False, x3=0):
        s, l = slogpf(A, skew)
        f = (s * l.exp())[:, None, None] if adjugate else 1.0
        return s, l, _out(f * torch.linalg.inv(_skew(A.detach(), skew)))

    def slogpf_factors(A, skew):
        return (*slogpf(A, skew), _out(_skew(A.detach(), skew)), A.new_zeros(A.shape[0], A.shape[-1] // 2),
                torch.zeros(A.shape[:-1], dtype=torch.int32))

    def slogpf_inverse(gbuf, d, perm, n, scale=None, x3=0):
        _raw(gbuf, d, perm, scale)
        return _out(scale[:, None, None] * torch.linalg.inv(gbuf))

    for f in (slogdet, slogdet_parts, slogdet_factors, slogdet_inverse, det_parts, slogpf, slogpf_parts,
              slogpf_factors, slogpf_inverse):
        mp.setattr(_kernels, f.__name__, f)
    # the library's choice of a kernel family, without the library's state
    mp.setattr(_diff._tune, "kernel_family", lambda n, op: "fused")


def _matrix(n, op, dt, device="cpu"):
    g = torch.Generator().manual_seed(7 * n)
    A = 0.25 * torch.randn(3, n, n, generator=g, dtype=dt) / n**0.5
    J = torch.eye(n, dtype=dt)
    if op in ("slogpf", "pf"):
        J = torch.kron(torch.eye(n // 2), torch.tensor([[0.0, 1.0], [-1.0, 0.0]])).to(dt)
    return (A + J).to(device)


def _value(out):
    return out[1] if isinstance(out, tuple) else out


def _under(transform, f, W, t):
    """f's value of the closed-over W, through a transform of something else."""
    if transform == "vmap":
        return torch.vmap(lambda x: x * _value(f(W)).sum())(t).sum()
    if transform == "grad":
        return torch.func.grad(lambda x: (x * _value(f(W)).sum()).sum())(t).sum()
    if transform == "jvp":
        return torch.func.jvp(lambda x: x * _value(f(W)).sum(), (t,), (torch.ones_like(t),))[1].sum()
    return torch.vmap(torch.func.grad(lambda x: x * _value(f(W)).sum()))(t).sum()


CASES = [(op, n, dt) for op in ("slogdet", "slogpf", "det", "pf") for n, dt in (
    (6, torch.float32), (34, torch.float32), (6, torch.float64), (34, torch.float64))]
TRANSFORMS = ["vmap", "grad", "jvp", "vmap_grad"]


def check(f, op, n, dt, transform, requires, device="cpu"):
    W = _matrix(n, op, dt, device).requires_grad_(requires)
    t = torch.tensor([0.5, 2.0], dtype=dt, device=device)
    want = _value(f(W)).sum() * (t.sum() if transform == "vmap" else t.numel())
    got = _under(transform, f, W, t)
    assert torch.equal(got, want) or abs(got - want) <= 8 * torch.finfo(dt).eps * abs(want)
    assert got.requires_grad == requires
    if requires:
        (g,) = torch.autograd.grad(got, W)
        (r,) = torch.autograd.grad(want, W)
        assert torch.linalg.vector_norm(g - r) <= 8 * n * torch.finfo(dt).eps * torch.linalg.vector_norm(r)


@pytest.mark.parametrize("requires", [False, True])
@pytest.mark.parametrize("transform", TRANSFORMS)
@pytest.mark.parametrize("op,n,dt", CASES)
def test_closed_over(monkeypatch, op, n, dt, transform, requires):
    _stub(monkeypatch)
    f = (lambda A: getattr(_diff, op)(A, True)) if op in ("slogpf", "pf") else getattr(_diff, op)
    check(f, op, n, dt, transform, requires)


@pytest.mark.gpu
@pytest.mark.parametrize("requires", [False, True])
@pytest.mark.parametrize("transform", TRANSFORMS)
@pytest.mark.parametrize("op,n,dt", CASES)
def test_closed_over_on_the_gpu(dev, op, n, dt, transform, requires):
    print(f"closed over {op} n={n} {dt} {transform} {requires}", flush=True)
    check(getattr(fermix_amd, op), op, n, dt, transform, requires, dev)
