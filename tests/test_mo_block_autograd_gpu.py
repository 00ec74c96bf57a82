"""Derivatives with respect to the C1 of B_tensor_gen_block, which is linear in
it: backward and forward mode, as with a product of torch's."""

import pytest
import torch
import torch.autograd.forward_ad as fwad

from forte2_amd.jkbuilder import FockBuilder
from forte2_amd.workloads import orthonormal_C, synthetic_B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,N,n1,n2", [(40, 33, 7, 12), (40, 33, 12, 7), (9, 20, 45, 5)])
def test_derivatives_in_c1(dev, Q, N, n1, n2):
    print(f"[mo-grad] Q={Q} N={N} n1={n1} n2={n2}", flush=True)
    B = synthetic_B(Q, N, seed=1, device=dev)
    fb = FockBuilder(B=B, device=dev)
    g = torch.Generator(device=dev)
    g.manual_seed(3)
    C1 = torch.randn((N, n1), generator=g, device=dev, dtype=torch.float64)
    T = torch.randn((N, n1), generator=g, device=dev, dtype=torch.float64)
    W = torch.randn((Q, n1, n2), generator=g, device=dev, dtype=torch.float64)
    C2 = orthonormal_C(N, n2, seed=2, device=dev)
    plain = fb.B_tensor_gen_block(C1, C2)
    assert not plain.requires_grad
    X = torch.matmul(B, C2)  # (Q, N, n2)
    ref = torch.matmul(W, X.transpose(1, 2).contiguous()).sum(0).T  # d <W, out> / d C1
    tol = 1e-12 * float(ref.abs().max())
    # backward
    c = C1.clone().requires_grad_(True)
    out = fb.B_tensor_gen_block(c, C2)
    assert float((out - plain).abs().max()) <= 1e-12
    (out * W).sum().backward()
    assert float((c.grad - ref).abs().max()) <= tol
    # forward mode
    with fwad.dual_level():
        t = fwad.unpack_dual(fb.B_tensor_gen_block(fwad.make_dual(C1, T), C2)).tangent
    assert t is not None and float((t - torch.matmul(T.T.contiguous(), X)).abs().max()) <= 1e-12
    # without recording: the plain result, bitwise
    with torch.no_grad():
        assert torch.equal(fb.B_tensor_gen_block(c, C2), plain)
