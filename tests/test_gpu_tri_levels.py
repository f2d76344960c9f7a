"""The blocked float32 inverse's recursion levels at padded orders N below the power of two
they recurse to (tiles past N left out), and the two factors' levels on two streams (small
batches) against one (large ones): A^-T against float64, the members of a large batch equal
to the same members in a small one bit for bit."""

import numpy as np
import pytest
import torch

from fermix_amd import _kernels
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
