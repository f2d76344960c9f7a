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
