"""The blocked float32 inverse's recursion levels at padded orders N below the power of two
they recurse to (tiles past N left out), and the two factors' levels on two streams (small
batches) against one (large ones): A^-T against float64, the members of a large batch equal
to the same members in a small one bit for bit."""

import numpy as np
import pytest
import torch

from fermix_amd import _kernels, _lib
from tests.tolerances import relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,big", [(129, 520), (192, 520), (193, 520), (257, 136), (300, 136), (330, 136), (385, 136), (520, 40)])
@pytest.mark.parametrize("x3", [0, 1])
def test_levels(dev, n, big, x3):
    rng = np.random.default_rng(9300 + n)
    A = (np.eye(n) + 0.5 * rng.standard_normal((4, n, n)) / np.sqrt(n)).astype(np.float32)[:, rng.permutation(n)]
    print(f"tri levels n={n} x3={x3}", flush=True)
    At = torch.from_numpy(np.ascontiguousarray(A)).to(dev)
    inv = _kernels.slogdet_parts(At, x3=x3)[2]
    ref = np.linalg.inv(A.astype(np.float64)).swapaxes(1, 2)
    got = inv.cpu().numpy()
    # the members' condition numbers are below 10: 1e-4 is the repository's gradient bar
    assert max(relerr(got[k], ref[k]) for k in range(4)) < 1e-4
    many = At.repeat((big + 3) // 4, 1, 1)
    assert torch.equal(_kernels.slogdet_parts(many, x3=x3)[2][-4:], inv)


@pytest.mark.parametrize("n", [129, 193, 300, 520, 700, 1100])
@pytest.mark.parametrize("x3", [0, 1])
def test_stale_workspace(dev, n, x3):
    """The tiles that are left out stay unwritten in the workspace and in the output, which
    holds the upper factor's intermediate: the same bits over stale NaN as over zeros, with
    64- and 128-wide tiles (fp32 products take the wide ones from level 512 on)."""
    rng = np.random.default_rng(9350 + n)
    B = 3
    A = (np.eye(n) + 0.5 * rng.standard_normal((B, n, n)) / np.sqrt(n)).astype(np.float32)[:, rng.permutation(n)]
    print(f"stale workspace n={n} x3={x3}", flush=True)
    sign, _, lu0, perm = _kernels.slogdet_factors(torch.from_numpy(np.ascontiguousarray(A)).to(dev), x3)
    L = _lib.lib()
    wsb = L.fx_slogdet_inverse_f32_workspace(B, n)
    got = []
    for stale in (0.0, float("nan")):
        lu = lu0.clone()
        ws = torch.full((wsb // 4,), stale, device=dev)
        out = torch.full((B, n, n), stale, device=dev)
        st = L.fx_slogdet_inverse_f32(lu.data_ptr(), perm.data_ptr(), sign.data_ptr(), None, B, n, 1, out.data_ptr(), x3,
                                      ws.data_ptr(), wsb, torch.cuda.current_stream().cuda_stream or None)
        assert st == 0
        got.append(out)
    assert bool(torch.isfinite(got[0]).all()) and bool((got[0] != 0).any()) and torch.equal(*got)
