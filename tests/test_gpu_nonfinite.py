"""NaN, infinite and tiny members through the n <= 128 kernels: they end, they leave the other
members' bits alone (four members share a workgroup for n <= 32), a NaN shows in logabs and
the matrices behind the gradients stay finite; and members scaled by a power of two, down to
where the determinant underflows, give the unscaled member's sign and exactly scaled inverse."""

import numpy as np
import pytest
import torch

import fermix_amd
from fermix_amd import _kernels

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f64": torch.float64, "c64": torch.complex64, "c128": torch.complex128}
# |x|^2 of a complex pivot stays a normal number
SCALE = {"f32": 2.0**-60, "f64": 2.0**-900, "c64": 2.0**-50, "c128": 2.0**-400}


def _make(dev, kind, pf, n):
    g = torch.Generator(device=dev).manual_seed(17 * n)
    A = 0.25 * torch.randn(7, n, n, generator=g, device=dev, dtype=DT[kind]) / n**0.5
    J = torch.eye(n, device=dev, dtype=DT[kind])
    if pf:
        i = torch.arange(0, n, 2, device=dev)
        J = torch.zeros_like(J)
        J[i, i + 1], J[i + 1, i] = 1, -1
    A = (A - A.mT if pf else A) + J
    order = torch.randperm(n, generator=torch.Generator().manual_seed(n)).to(dev)
    return A[:, order][:, :, order].contiguous() if pf else A[:, order].contiguous()


def _parts(kind, pf, A):
    """(sign, logabs, inverse) as the gradient forms them."""
    if pf:
        return _kernels.slogpf_parts(A, False)
    if kind == "f32" and A.shape[-1] > 32:
        s, l, lu, perm = _kernels.slogdet_factors(A)
        return s, l, _kernels.slogdet_inverse(lu, perm, s, A.shape[-1])
    return _kernels.slogdet_parts(A)[:3]


def _values(pf, A):
    return fermix_amd.slogpf(A, skew_symmetrize=False) if pf else fermix_amd.slogdet(A)


CASES = [(pf, n) for pf in (False, True) for n in (8, 32, 48, 64, 100, 128)] + [(False, 17), (False, 65)]


@pytest.mark.parametrize("kind", list(DT))
@pytest.mark.parametrize("pf,n", CASES)
def test_nonfinite(dev, kind, pf, n):
    A = _make(dev, kind, pf, n)
    bad = A.clone()
    nan, inf = float("nan"), float("inf")
    for b, entries in ((1, [(0, n - 1, nan)]), (3, [(n // 2, 1, inf)]), (5, [(n - 1, 0, inf), (n // 2, 2, nan)])):
        for i, j, v in entries:
            bad[b, i, j] = v
            if pf:
                bad[b, j, i] = -v
    print(f"nonfinite {kind} pf={pf} n={n}", flush=True)
    good = [0, 2, 4, 6]
    for f in (lambda X: _values(pf, X), lambda X: _parts(kind, pf, X)):
        for x, y in zip(f(A), f(bad)):
            assert torch.equal(x[good], y[good])
    _, l = _values(pf, bad)
    assert bool(torch.isnan(l[[1, 5]]).all()) and not bool(torch.isfinite(l[3]))
    inv = _parts(kind, pf, bad)[2]
    assert bool(torch.isfinite(torch.view_as_real(inv) if inv.is_complex() else inv).all())


@pytest.mark.parametrize("kind", list(DT))
@pytest.mark.parametrize("pf,n", CASES)
def test_scaled(dev, kind, pf, n):
    A = _make(dev, kind, pf, n)
    c = SCALE[kind]
    print(f"scaled {kind} pf={pf} n={n}", flush=True)
    s, l, inv = _parts(kind, pf, A)
    t, m, jnv = _parts(kind, pf, A * c)
    shift = (n // 2 if pf else n) * np.log(c)
    eps = torch.finfo(DT[kind]).eps
    assert bool((inv != 0).any())
    if kind == "f32" and pf:  # its formula replaces the smallest pivot by 1: not scale-free
        assert torch.linalg.vector_norm(inv - jnv * c) <= 1e-4 * torch.linalg.vector_norm(inv)
    else:
        assert torch.equal(inv, jnv * c)
    assert bool((abs(t - s) <= 2 * eps).all())
    # the logs are summed at the size of the shift
    assert bool((abs(m - (l + shift)) <= n * eps * abs(shift)).all())
    for x, y in zip(_values(pf, A * c), (t, m)):
        assert torch.equal(x, y)
