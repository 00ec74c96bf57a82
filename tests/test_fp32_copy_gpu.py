"""The FP32 copy that FockBuilder.B_fp32 hands out may be written in place (its
zero pattern stays): the next build, and a replay of a captured one, use the
new values in J as in K."""

import pytest
import torch

from forte2_amd.jkbuilder import FockBuilder
from forte2_amd.workloads import orthonormal_C, synthetic_B

pytestmark = pytest.mark.gpu


def _banded(dev, Q, N, keep):
    B = synthetic_B(Q, N, seed=N, device=dev)
    i = torch.arange(N, device=dev)
    return B.mul_(((i[:, None] - i[None, :]).abs() < keep).to(B.dtype))


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("inference", [False, True])
def test_values_written_in_place(dev, prec, inference):
    Q, N = 45, 64
    print(f"[fp32-copy] {prec} inference={inference}", flush=True)
    C = orthonormal_C(N, 5, seed=2, device=dev)
    with torch.inference_mode(inference):
        fb = FockBuilder(B=_banded(dev, Q, N, 6), device=dev, precision=prec)
        fb.build_JK([C])
        fb.B_fp32().mul_(3.0).add_(fb.B_fp32().roll(1, 0))
        J, K = fb.build_JK([C])
        Jd = fb.build_J([C @ C.T])
        ref = FockBuilder(B=fb.B_fp32().to(torch.float64), device=dev, precision=prec, j_sparse=False)
        Jr, Kr = ref.build_JK([C])
    # FP64 sums of the same products, in another order
    assert float((J[0] - Jr[0]).abs().max()) <= 1e-12 * float(Jr[0].abs().max())
    assert float((Jd[0] - Jr[0]).abs().max()) <= 1e-12 * float(Jr[0].abs().max())
    assert torch.equal(K[0], Kr[0])


def test_replay_after_a_write_in_place(dev):
    Q, N = 45, 64
    fb = FockBuilder(B=_banded(dev, Q, N, 6), device=dev, precision="bf16x3")
    C = orthonormal_C(N, 5, seed=2, device=dev)
    fb.build_JK([C])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        J, K = fb.build_JK([C])
    for k in range(3):
        fb.B_fp32().mul_(1.5)
        graph.replay()
        torch.cuda.synchronize()
        got = J[0].clone(), K[0].clone()
        ref = fb.build_JK([C])  # eager work between the replays
        torch.cuda.synchronize()
        assert torch.equal(got[0], ref[0][0]) and torch.equal(got[1], ref[1][0])
