"""The one-launch gradient kernels of the orders n <= 128 (small_inverse.hip) at the edges of
their 16-column blocks, through the C ABI's factor -> inverse calls and the adjugates:
odd and even numbers of blocks, n = N and n < N, n with and without 16-byte rows, batches
that leave a workgroup of four partly empty; with a per-member scale, and with members
that have one, two and more exact zero pivots. References in float64: numpy's inverse, the
SVD adjugate and the oracle's Pfaffian adjugate run in float64.

Bar: 1e-4 relative Frobenius error, the repository's float32 gradient bar; the members are
I (or J) + noise of norm 1/2, condition numbers below 10, for which a backward-stable
float32 inverse errs by at most about n 2^-24 kappa = 8e-5 at n = 128."""

import numpy as np
import pytest
import torch

from fermix_amd import _kernels
from oracle import generic as g
from oracle import ref64
from tests.tolerances import relerr

pytestmark = pytest.mark.gpu

ORDERS = [1, 2, 15, 16, 17, 31, 32, 33, 48, 50, 64, 66, 79, 80, 82, 96, 97, 111, 112, 114, 127, 128]


def _t(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


def _close(got, ref, what):
    for k in range(ref.shape[0]):
        if np.abs(ref[k]).max() == 0:
            assert np.all(got[k] == 0), (what, k)
        else:
            assert relerr(got[k], ref[k]) < 1e-4, (what, k, relerr(got[k], ref[k]))


@pytest.mark.parametrize("n", ORDERS)
def test_lu(dev, n):
    B = 7
    rng = np.random.default_rng(8800 + n)
    A = (np.eye(n) + 0.5 * rng.standard_normal((B, n, n)) / np.sqrt(n)).astype(np.float32)
    A = A[:, rng.permutation(n)]
    w = rng.uniform(0.5, 2.0, B).astype(np.float32)
    print(f"lu inverse n={n}", flush=True)
    s, _, lu, perm = _kernels.slogdet_factors(_t(A, dev))
    got = _kernels.slogdet_inverse(lu, perm, s, n, scale=_t(w, dev)).cpu().numpy()
    _close(got, w[:, None, None] * np.linalg.inv(A.astype(np.float64)).swapaxes(1, 2), f"inverse n={n}")
    A[1, :, n // 2] = 0.0  # one zero pivot
    A[2, n - 1] = 0.0
    A[3, :, 0] = 0.0
    A[3, n // 2] = 0.0  # two zero pivots, rank n - 1
    A[4, :, : min(n, 3)] = 0.0
    s, _, lu, perm = _kernels.slogdet_factors(_t(A, dev))
    got = _kernels.slogdet_inverse(lu, perm, s, n).cpu().numpy()
    assert np.all(got[1:5] == 0) and np.all(np.isfinite(got))
    ref = np.stack([ref64.adjT_svd(a) for a in A])
    ref[4] = 0.0 if n > 1 else ref[4]
    _close(_kernels.det_parts(_t(A, dev))[2].cpu().numpy(), ref, f"adjugate n={n}")


@pytest.mark.parametrize("n", [n for n in ORDERS if n % 2 == 0])
def test_pf(dev, n):
    B = 5
    rng = np.random.default_rng(8900 + n)
    J = np.kron(np.eye(n // 2), np.array([[0.0, 1.0], [-1.0, 0.0]]))
    X = rng.standard_normal((B, n, n)) / np.sqrt(n)
    order = rng.permutation(n)
    S = (J + 0.25 * (X - X.swapaxes(1, 2)))[:, order][:, :, order].astype(np.float32)
    w = rng.uniform(0.5, 2.0, B).astype(np.float32)
    print(f"pf inverse n={n}", flush=True)
    _, _, gbuf, d, perm = _kernels.slogpf_factors(_t(S, dev), False)
    got = _kernels.slogpf_inverse(gbuf, d, perm, n, scale=_t(w, dev)).cpu().numpy()
    assert np.array_equal(got, -got.swapaxes(1, 2))
    _close(got, w[:, None, None] * np.linalg.inv(S.astype(np.float64)), f"inverse n={n}")
    for k, rows in ((1, [n // 2]), (2, [0, n - 1]), (3, list(range(min(n, 4))))):
        S[k, rows] = 0.0  # one zero pivot, two (the lifted evaluation for n > 2), more
        S[k][:, rows] = 0.0
    _, _, gbuf, d, perm = _kernels.slogpf_factors(_t(S, dev), False)
    got = _kernels.slogpf_inverse(gbuf, d, perm, n).cpu().numpy()
    assert np.all(got[1:4] == 0) and np.all(np.isfinite(got))
    ref = g.pf_parts_generic(S.astype(np.float64), True)[2]
    _close(_kernels.slogpf_parts(_t(S, dev), False, adjugate=True)[2].cpu().numpy(), ref, f"adjugate n={n}")


@pytest.mark.parametrize("n", [8, 16, 32, 33, 64, 100, 128])
def test_det_scale(dev, n):
    """adj(A)^T of diagonal matrices of powers of two is exact in float32, inverse and
    determinant alike: one rounding at most is left, where exp of a float32 logabs gave up to
    2^-25 logabs, 6e-7 at n = 32."""
    rng = np.random.default_rng(8950 + n)
    d = rng.choice(np.array([2.0, -2.0, 1.0, 4.0, 0.5]), (24, n))
    order = rng.permutation(n)
    A = np.zeros((24, n, n), np.float32)
    A[:, np.arange(n), order] = d
    print(f"det scale n={n}", flush=True)
    adj = _kernels.det_parts(_t(A, dev))[2].cpu().numpy().astype(np.float64)
    det = np.prod(d, axis=1) * np.linalg.det(np.eye(n)[:, order])
    ref = np.zeros(A.shape)
    ref[:, np.arange(n), order] = det[:, None] / d
    assert np.all(adj[ref == 0] == 0)
    err = np.abs(adj[ref != 0] - ref[ref != 0]) / np.abs(ref[ref != 0])
    assert np.max(err) <= 2.0**-24, np.max(err)


def _f32(x):
    return x.astype(np.float32)


def _pf_inverse(gbuf, d, perm):
    """S^-1 from the Parlett-Reid factors in float32, every sum in one chain of fma: L~, its
    inverse Y by substitution, R = Y^T D~^-1 Y and the rank-2 correction."""
    B, N = perm.shape
    at, f = np.arange(B)[:, None], np.arange(N)
    G = gbuf.transpose(0, 2, 1, 3).reshape(B, N, N)[at, perm]  # by position
    K = np.abs(d).argmin(1)
    dt = d.copy()
    dt[at[:, 0], K] = 1
    L = np.empty_like(G)
    L[:, :, 0::2] = _f32(G[:, :, 1::2] * _f32(1 / dt)[:, None, :])
    L[:, :, 1::2] = G[:, :, 0::2]
    L[:, f[:, None] <= (f | 1)[None, :]] = 0
    Y = np.broadcast_to(np.eye(N, dtype=np.float32), G.shape).copy()
    for t in range(N):
        Y[:, t + 1 :] = _f32(Y[:, t + 1 :] - np.float64(L[:, t + 1 :, t, None]) * Y[:, t, None, :])
    DY = np.empty_like(Y)
    DY[:, 0::2] = _f32(Y[:, 1::2] * _f32(1 / dt)[:, :, None])
    DY[:, 1::2] = -_f32(Y[:, 0::2] * _f32(1 / dt)[:, :, None])
    R = np.zeros_like(Y)
    for t in range(N):
        R = _f32(R + np.float64(Y[:, t, :, None]) * DY[:, t, None, :])
    R = np.tril(R, -1)
    R = R - R.transpose(0, 2, 1)
    dK, w, v = d[at[:, 0], K], R[at[:, 0], :, 2 * K], Y[at[:, 0], 2 * K]
    a2 = _f32((1 - dK) / dK)
    R = -_f32(R + a2[:, None, None] * _f32(_f32(w[:, :, None] * v[:, None, :]) - _f32(v[:, :, None] * w[:, None, :])))
    out = np.empty_like(R)
    out[at[:, :, None], perm[:, :, None], perm[:, None, :]] = R
    return out


@pytest.mark.parametrize("n", [16, 32, 64, 96, 128])
def test_pf_error_of_the_unblocked_inverse(dev, n):
    """S^-1 against substitution and products that round every term into one running sum: the
    geometric mean over the members of the errors' ratio (its scatter is below 0.01). Bar
    0.945: the inverse by 32 x 32 leaves and GEMMs that this kernel took the place of has 0.92
    to 0.942 at these orders."""
    B = 2048 // n * 4
    rng = np.random.default_rng(8970 + n)
    # the pairing of neighbouring standing waves at sites in a random order with random signs
    i = np.arange(n)
    C = np.cos((i[:, None] + 0.5) * i * (np.pi / n)) * np.sqrt(2.0 / n)
    C[:, 0] /= np.sqrt(2.0)
    Q = C[:, 0::2] @ C[:, 1::2].T
    Q = Q - Q.T
    order = rng.permuted(np.tile(i, (B, 1)), axis=1)
    sign = rng.choice([-1.0, 1.0], (B, n))
    Q = Q[order[:, :, None], order[:, None, :]] * sign[:, :, None] * sign[:, None, :]
    X = rng.standard_normal((B, n, n)) / np.sqrt(n)
    S = _f32(1.5 * (Q + 0.25 * (X - X.swapaxes(1, 2))))
    S = (S - S.swapaxes(1, 2)) / 2
    print(f"pf error n={n}", flush=True)
    _, _, gbuf, d, perm = _kernels.slogpf_factors(_t(S, dev), False)
    got = _kernels.slogpf_inverse(gbuf, d, perm, n).cpu().numpy()
    bar = _pf_inverse(gbuf.cpu().numpy(), d.cpu().numpy(), perm.cpu().numpy())
    want = np.linalg.inv(S.astype(np.float64))
    e, b = (np.sqrt(np.sum((x - want) ** 2, axis=(1, 2))) for x in (got, bar))
    ratio = float(np.exp(np.mean(np.log(e / b))))
    print("error, as a multiple:", ratio, flush=True)
    assert ratio <= 0.945
