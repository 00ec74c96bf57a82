"""Sizes at which one thread per element, row or P would be more threads than a
launch can count (2^32 in a dimension): the launches split there, and every
output is written.  The values are chosen so that every sum is exact."""

import pytest
import torch

from forte2_amd.jkbuilder import FockBuilder

pytestmark = pytest.mark.gpu


def test_half_transform_of_2_30_rows(dev):
    # nbf 1: four threads a row
    Q = (1 << 30) + 3
    print(f"[launch-limits] half-transform, {Q} rows", flush=True)
    B = torch.arange(Q, dtype=torch.float64, device=dev).view(Q, 1, 1)
    fb = FockBuilder(B=B, device=dev, j_sparse=False)
    X = fb.half_transform(torch.full((1, 1), 2.0, dtype=torch.float64, device=dev))
    assert torch.equal(X, B.mul_(2.0))
    fb.release()


def test_gamma_of_2_25_p(dev):
    # nbf 1, two densities: a wave per density and P
    Q = (1 << 25) + 5
    print(f"[launch-limits] gamma, {Q} P", flush=True)
    B = torch.zeros(Q, dtype=torch.float64, device=dev)
    B[::4097], B[-1] = 2.0, 3.0
    n = -(-Q // 4097)
    fb = FockBuilder(B=B.view(Q, 1, 1), device=dev, j_sparse=False)
    C = [torch.full((1, 1), x, dtype=torch.float64, device=dev) for x in (1.0, 2.0)]
    J, K = fb.build_JK(C)
    ref = 4.0 * n + (9.0 if (Q - 1) % 4097 else 5.0)
    for d, f in enumerate((1.0, 4.0)):
        assert float(J[d]) == f * ref and float(K[d]) == f * ref
    fb.release()


def test_k_reduction_of_nbf_32772(dev):
    N = 32772
    print(f"[launch-limits] K, nbf {N}", flush=True)
    x = torch.arange(N, dtype=torch.float64, device=dev) % 1024
    B = torch.zeros((1, N, N), dtype=torch.float64, device=dev)
    B[0].diagonal().copy_(x)
    fb = FockBuilder(B=B, device=dev, j_sparse=False)
    K = fb.build_K([torch.ones((N, 1), dtype=torch.float64, device=dev)])[0]
    assert torch.equal(K, torch.outer(x, x))
    fb.release()


def test_j_reduction_of_nbf_46343(dev):
    # odd: one element per thread group
    N = 46343
    print(f"[launch-limits] J, nbf {N}", flush=True)
    r = torch.arange(N, dtype=torch.float64, device=dev) % 512 + 1.0
    B = (r[:, None] + r[None, :]).view(1, N, N)
    D = torch.zeros((N, N), dtype=torch.float64, device=dev)
    D[0, 0] = 1.0
    fb = FockBuilder(B=B, device=dev, j_sparse=False)
    J = fb.build_J([D])[0]
    del D
    assert torch.equal(J, B[0].mul_(2.0))  # gamma = B[0, 0, 0] = 2
    fb.release()
    torch.cuda.empty_cache()
