"""J/K at the edges of the split reductions: sizes around the 4 x 16 blocks of
the K reduction and the 64 elements of the J reduction, fewer splits than the
four waves that share them, and a B that is zero throughout.

Tolerance: FP64 sums of at most Q * nocc products of O(0.05)^2 values; the
rounding of such a sum is below 1e-12, the bar of the plain form is 1e-10.
"""

import numpy as np
import pytest
import torch

from forte2_amd.jkbuilder import FockBuilder
from forte2_amd.workloads import orthonormal_C, synthetic_B
from oracle import jk as ojk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("Q,N,noccs", [(1, 1, [1]), (3, 2, [1, 1]), (5, 4, [2]), (2, 15, [3]), (139, 16, [4]), (7, 17, [5, 4]),
                                       (40, 31, [6]), (33, 128, [9]), (65, 129, [10, 9])])
def test_reductions(dev, Q, N, noccs, sparse):
    print(f"[reductions] Q={Q} N={N} nocc={noccs} sparse={sparse}", flush=True)
    B = synthetic_B(Q, N, seed=Q + N, device=dev)
    Cs = [orthonormal_C(N, o, seed=N + k, device=dev) for k, o in enumerate(noccs)]
    J, K = FockBuilder(B=B, device=dev, j_sparse=sparse).build_JK(Cs)
    Jr, Kr = ojk.build_JK(B.cpu().numpy(), [c.cpu().numpy() for c in Cs])
    for k in range(len(noccs)):
        assert np.abs(J[k].cpu().numpy() - Jr[k]).max() <= 1e-10
        assert np.abs(K[k].cpu().numpy() - Kr[k]).max() <= 1e-10
        assert torch.equal(J[k], J[k].T) and torch.equal(K[k], K[k].T)


def test_zero_tensor(dev):
    B = torch.zeros((9, 20, 20), dtype=torch.float64, device=dev)
    C = orthonormal_C(20, 4, seed=1, device=dev)
    fb = FockBuilder(B=B, device=dev)
    for prec in ("fp64", "bf16x3"):
        J, K = fb.build_JK([C], precision=prec)
        assert float(J[0].abs().max()) == 0.0 and float(K[0].abs().max()) == 0.0


@pytest.mark.parametrize("N,keep", [(7, 3), (36, 12), (64, 4), (130, 40)])
def test_packed_elements_give_the_same_j(dev, N, keep):
    # the J passes over the packed nonzero elements of the FP32 copy read the
    # same elements in the same order: bitwise J, for J from C and from D
    Q = 45
    B = synthetic_B(Q, N, seed=N, device=dev)
    i = torch.arange(N, device=dev)
    B.mul_(((i[:, None] - i[None, :]).abs() < keep).to(B.dtype))
    C = orthonormal_C(N, 3, seed=2, device=dev)
    out = []
    for pack in (0, 1):
        fb = FockBuilder(B=B, device=dev, precision="bf16x3")
        fb.set_tuning("j_pack", pack)
        out.append(fb.build_JK([C])[0] + fb.build_J([C @ C.T]))
    assert all(torch.equal(a, b) for a, b in zip(*out))
