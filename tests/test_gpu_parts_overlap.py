"""slogpf + S^-1 of float64 and complex with the Parlett-Reid on a second stream beside the LU
(n <= 512): the bits of the unsplit run, which a captured graph takes, over several replays
with eager work on the same inputs in between."""

import pytest
import torch

from fermix_amd import _kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float64, torch.complex64, torch.complex128])
@pytest.mark.parametrize("n", [130, 302])
def test_overlap_is_the_captured_run(dev, dt, n):
    g = torch.Generator(device=dev).manual_seed(n)
    A = torch.randn(5, n, n, generator=g, device=dev, dtype=dt)
    A[3, 7] = A[3, :, 7] = 0
    B = torch.randn(5, n, n, generator=g, device=dev, dtype=dt)
    print(f"parts overlap {dt} n={n}", flush=True)
    want = {0: _kernels.slogpf_parts(A, True), 1: _kernels.slogpf_parts(B, True)}
    X = A.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = _kernels.slogpf_parts(X, True)
    for k in (0, 1, 0, 1):
        X.copy_(A if k == 0 else B)
        graph.replay()
        eager = _kernels.slogpf_parts(X, True)
        torch.cuda.synchronize()
        for a, b, c in zip(got, want[k], eager):
            assert torch.equal(a, b) and torch.equal(c, b)
    assert torch.all(want[0][2][3] == 0) and want[0][0][3] == 0
