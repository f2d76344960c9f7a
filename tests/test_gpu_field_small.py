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


def _fma(r, l, p):
    """r - l p as the unblocked kernels round it: one fma, or for complex two a component."""
    x = np.longdouble
    if not np.iscomplexobj(r):
        return (r - x(l) * x(p)).astype(r.dtype)
    re = (x(r.real) + x(l.imag) * x(p.imag)).astype(r.real.dtype)
    im = (x(r.imag) - x(l.imag) * x(p.real)).astype(r.real.dtype)
    re, im = re - x(l.real) * x(p.real), im - x(l.real) * x(p.imag)
    return re.astype(r.real.dtype) + 1j * im.astype(r.real.dtype)


def _elimination(A):
    """(sign, logabs, A^-T) by unblocked Gauss-Jordan on [A | I] in A's own precision: the pivot
    of largest |re| + |im|, one update of every entry a column, the logs and phases of the
    pivots taken one by one."""
    B, n, _ = A.shape
    at = np.arange(B)
    M = np.concatenate([A, np.broadcast_to(np.eye(n, dtype=A.dtype), A.shape)], axis=2)
    free = np.ones((B, n), bool)
    row = np.zeros((B, n), int)
    sign, logabs = np.ones(B, A.dtype), np.zeros(B, A.real.dtype)
    for j in range(n):
        row[:, j] = p = np.where(free, np.abs(M[:, :, j].real) + np.abs(M[:, :, j].imag), -1).argmax(1)
        free[at, p] = False
        P, d = M[at, p].copy(), M[at, p, j]
        sign, logabs = sign * (d / np.abs(d)), logabs + np.log(np.abs(d))
        l = M[:, :, j] * (1 / d)[:, None]
        l[at, p] = 0
        M[:, :, j + 1 :] = _fma(M[:, :, j + 1 :], l[:, :, None], P[:, None, j + 1 :])
    inv = np.stack([M[at, row[:, j], n:] / M[at, row[:, j], j][:, None] for j in range(n)], axis=1)
    return sign * _parity(row), logabs, inv.swapaxes(1, 2)


def _parity(row):
    """The sign of each row's permutation (its columns' inversions)."""
    return np.array([(-1.0) ** sum(int(np.sum(r[:k] > r[k])) for k in range(len(r))) for r in row])


def _true(A):
    """(sign, logabs, A^-T) in 80-bit arithmetic."""
    a = A.astype(np.clongdouble if np.iscomplexobj(A) else np.longdouble)
    B, n, _ = a.shape
    at = np.arange(B)
    U, sign, logabs = a.copy(), np.ones(B, a.dtype), np.zeros(B, np.longdouble)
    for k in range(n):
        p = k + np.abs(U[:, k:, k]).argmax(1)
        r = U[at, p].copy()
        U[at, p] = U[:, k]
        U[:, k] = r
        d = r[:, k]
        sign, logabs = np.where(p == k, sign, -sign) * d / np.abs(d), logabs + np.log(np.abs(d))
        U[:, k + 1 :, k + 1 :] -= (U[:, k + 1 :, k] / d[:, None])[:, :, None] * r[:, None, k + 1 :]
    X = np.linalg.inv(_wide(A)).astype(a.dtype)
    for _ in range(2):
        X = X + X @ (np.eye(n) - a @ X)
    return sign, logabs, X.swapaxes(1, 2)


@pytest.mark.parametrize("kind,n,B", [("f64", 63, 60), ("f64", 100, 30), ("c128", 64, 40), ("c128", 90, 20)])
def test_error_of_the_unblocked_elimination(dev, kind, n, B):
    """Blocked, and with the block's transformation formed explicitly, these kernels are no
    further from the exact results than the elimination that they stand for: the inverse as
    the geometric mean over the members of the errors' ratio (its scatter is 0.01), the sign
    and logabs, one value a member, as the errors' root mean square."""
    dt, _ = DT[kind]
    rng = np.random.default_rng(9500 + n)
    Q = np.linalg.qr(_noise(rng, (B, n, n), dt))[0]
    A = np.ascontiguousarray((1.5 * (Q + 0.5 * _noise(rng, (B, n, n), dt) / np.sqrt(n))).astype(dt))
    print(f"field_small error {kind} n={n}", flush=True)
    want = _true(A)

    def errors(got):
        s, l, i = (np.abs(g - w).astype(np.float64) for g, w in zip(got, want))
        return np.sqrt(np.mean(s**2)), np.sqrt(np.mean(l**2)), np.sqrt(np.sum(i**2, axis=(1, 2)))

    es, el, ei = errors([_np(x) for x in _kernels.slogdet_parts(torch.from_numpy(A).to(dev))[:3]])
    bs, bl, bi = errors(_elimination(A))
    ratio = float(np.exp(np.mean(np.log(ei / bi))))
    print("error, as a multiple: sign", es / max(bs, 1e-300), "logabs", el / bl, "inverse", ratio, flush=True)
    assert es <= bs and el <= bl and ratio <= 1.0
