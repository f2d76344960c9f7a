"""The LDS-resident LU / inverse and Parlett-Reid of float64, complex64 and complex128
(field_small.inc) at the edges of their 16-column panels, of the one- and two-row-per-lane
panels (n = 64 / 65), of the one-wave kernels (n = 32 / 33) and of the orders they cover
(complex128 LU n = 96 / 97): values against numpy in double, A^-T and S^-1 against numpy's
inverse, the skew-symmetrising load, exactly singular members, and the gradient call's
sign / logabs equal to the value's, bit for bit.

Bars: 4 n u kappa_2 relative Frobenius error for the inverses and 4 n u kappa_2 absolute for
logabs and the sign (u = 2^-53, 2^-24 for complex64), the first-order bound of a
backward-stable elimination with modest growth; the members are a permuted identity (or J)
plus noise of norm 1/2, kappa_2 below 10."""

import numpy as np
import pytest
import torch

import fermix_amd
from fermix_amd import _kernels
from oracle import ref64

pytestmark = pytest.mark.gpu

DT = {"f64": (np.float64, 2.0**-53), "c64": (np.complex64, 2.0**-24), "c128": (np.complex128, 2.0**-53)}
ORDERS = [1, 2, 15, 16, 17, 31, 32, 33, 48, 50, 63, 64, 65, 80, 81, 96, 97, 112, 113, 127, 128]


def _noise(rng, shape, dt):
    x = rng.standard_normal(shape)
    if np.issubdtype(dt, np.complexfloating):
        x = (x + 1j * rng.standard_normal(shape)) / np.sqrt(2.0)
    return x


def _wide(x):
    return x.astype(np.complex128 if np.iscomplexobj(x) else np.float64)


def _grid(x):
    """x on a grid of 2^-12, so that sums with small integers are exact in every type."""
    return (np.round(x * 2**12) / 2**12).astype(x.dtype)


def _np(x):
    return x.detach().cpu().numpy()


def _bar(x, n, u):
    return 4.0 * n * u * max(1.0, float(np.max([np.linalg.cond(m) for m in x])))


@pytest.mark.parametrize("kind", ["f64", "c64", "c128"])
@pytest.mark.parametrize("n", ORDERS)
def test_lu(dev, kind, n):
    dt, u = DT[kind]
    B = 6
    rng = np.random.default_rng(9100 + n)
    A = (np.eye(n) + 0.5 * _noise(rng, (B, n, n), dt) / np.sqrt(n)).astype(dt)[:, rng.permutation(n)]
    A[4, :, n // 2] = 0
    reg = [0, 1, 2, 3, 5]
    bar = _bar(_wide(A[reg]), n, u)
    print(f"field_small lu {kind} n={n}", flush=True)
    At = torch.from_numpy(np.ascontiguousarray(A)).to(dev)
    s, l = map(_np, fermix_amd.slogdet(At))
    s64, l64 = np.linalg.slogdet(_wide(A))
    assert s[4] == 0 and np.isneginf(l[4])
    assert np.max(np.abs(s[reg] - s64[reg])) <= bar and np.max(np.abs(l[reg] - l64[reg])) <= bar
    sp, lp, inv = map(_np, _kernels.slogdet_parts(At)[:3])
    assert np.array_equal(sp, s) and np.array_equal(lp, l)
    ref = np.linalg.inv(_wide(A[reg])).swapaxes(1, 2)
    err = np.linalg.norm(inv[reg] - ref, axis=(1, 2)) / np.linalg.norm(ref, axis=(1, 2))
    assert np.all(inv[4] == 0) and np.max(err) <= bar, (np.max(err), bar)
    sd, ld, adj = map(_np, _kernels.det_parts(At))
    assert np.array_equal(sd, s) and np.array_equal(ld, l)
    ref = np.stack([ref64.adjT_svd(a) for a in A])
    err = np.linalg.norm(adj - ref, axis=(1, 2)) / np.linalg.norm(ref, axis=(1, 2))
    assert np.max(err) <= 4 * bar, (np.max(err), bar)


@pytest.mark.parametrize("kind", ["f64", "c64", "c128"])
@pytest.mark.parametrize("n", [n for n in ORDERS if n % 2 == 0])
def test_pr(dev, kind, n):
    dt, u = DT[kind]
    B = 6
    rng = np.random.default_rng(9200 + n)
    J = np.kron(np.eye(n // 2), np.array([[0.0, 1.0], [-1.0, 0.0]]))
    X = _noise(rng, (B, n, n), dt) / np.sqrt(n)
    order = rng.permutation(n)
    S = (J + 0.25 * (X - X.swapaxes(1, 2)))[:, order][:, :, order].astype(dt)
    S = (S - S.swapaxes(1, 2)) / dt(2)
    S[4, n // 2] = 0
    S[4, :, n // 2] = 0
    reg = [0, 1, 2, 3, 5]
    bar = _bar(_wide(S[reg]), n, u)
    print(f"field_small pr {kind} n={n}", flush=True)
    St = torch.from_numpy(np.ascontiguousarray(S)).to(dev)
    s, l = map(_np, fermix_amd.slogpf(St, skew_symmetrize=False))
    pf = np.array([ref64.pf64(x) for x in S[reg]])
    assert s[4] == 0 and np.isneginf(l[4])
    assert np.max(np.abs(s[reg] - pf / np.abs(pf))) <= bar
    assert np.max(np.abs(l[reg] - np.log(np.abs(pf)))) <= bar
    sp, lp, inv = map(_np, _kernels.slogpf_parts(St, False)[:3])
    assert np.array_equal(sp, s) and np.array_equal(lp, l)
    ref = np.linalg.inv(_wide(S[reg]))
    err = np.linalg.norm(inv[reg] - ref, axis=(1, 2)) / np.linalg.norm(ref, axis=(1, 2))
    assert np.all(inv[4] == 0) and np.max(err) <= bar, (np.max(err), bar)
    # the skew part of S + (symmetric) is S: x - y and x + y are exact for these values
    Y = np.round(_noise(rng, (B, n, n), dt).real * 4).astype(dt)
    At = torch.from_numpy(np.ascontiguousarray(_grid(S) + (Y + Y.swapaxes(1, 2)))).to(dev)
    Bt = torch.from_numpy(np.ascontiguousarray(_grid(S))).to(dev)
    for got, want in zip(_kernels.slogpf_parts(At, True), _kernels.slogpf_parts(Bt, False)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("n", [16, 32, 33, 64, 65, 128])
def test_det_scale_c64(dev, n):
    """adj(A)^T = det A^-T with the det that the factorisation holds in double: of diagonal
    matrices of 2, -2, 2i, 1 the inverse and the adjugate are exact in complex64, and one
    rounding (2^-23 with the exp and the product) is left. A logabs rounded to float32 alone
    would give up to 2^-25 logabs, 1.3e-6 at n = 64."""
    rng = np.random.default_rng(9400 + n)
    d = rng.choice(np.array([2, -2, 2j, 1]), (24, n))
    A = np.zeros((24, n, n), np.complex64)
    A[:, np.arange(n), np.arange(n)] = d
    order = rng.permutation(n)
    A = A[:, order]
    print(f"field_small det scale n={n}", flush=True)
    adj = _np(_kernels.det_parts(torch.from_numpy(A).to(dev))[2])
    det = np.prod(d, axis=1) * np.linalg.det(np.eye(n)[order])
    ref = np.zeros(A.shape, np.complex128)
    ref[:, np.arange(n), order] = det[:, None] / d[:, order]
    assert np.all(adj[ref == 0] == 0)
    err = np.abs(adj[ref != 0] - ref[ref != 0]) / np.abs(ref[ref != 0])
    assert np.max(err) <= 2.0**-23, np.max(err)
