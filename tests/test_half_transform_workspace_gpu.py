"""f2jk_half_transform writes X where the caller wants it: its workspace holds
the packed coefficients only, and FockBuilder.half_transform allocates no more."""

import ctypes

import pytest
import torch

from forte2_amd import _native as nat
from forte2_amd.jkbuilder import FockBuilder
from forte2_amd.workloads import orthonormal_C, synthetic_B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,N,ncol", [(139, 24, 5), (300, 131, 21), (60, 340, 336)])
def test_workspace_holds_the_coefficients(dev, Q, N, ncol):
    print(f"[half-transform-ws] Q={Q} N={N} ncol={ncol}", flush=True)
    B = synthetic_B(Q, N, seed=Q, device=dev)
    C = orthonormal_C(N, ncol, seed=3, device=dev)
    fb = FockBuilder(B=B, device=dev, j_sparse=False)
    X = fb.half_transform(C)
    # whole tiles of 16 columns and 16 rows, at most 20 column blocks each
    cols = -(-ncol // 16) + 1
    assert fb._ws.numel() <= 8 * 16 * cols * (N + 16) + 256
    ref = torch.matmul(B.cpu(), C.cpu())
    assert float((X.cpu() - ref).abs().max()) <= 1e-12
    # one byte less is refused
    lib, size = nat.jk_lib(), ctypes.c_size_t()
    nat.jk_check(lib.f2jk_half_transform_workspace_size(fb.ctx, ncol, ctypes.byref(size)), "size")
    rc = lib.f2jk_half_transform(fb.ctx, ctypes.c_void_p(C.data_ptr()), ncol, ncol, 0, Q,
                                 ctypes.c_void_p(X.data_ptr()), ncol, nat.PREC["fp64"],
                                 ctypes.c_void_p(fb._ws.data_ptr()), size.value - 1, None)
    assert rc == -3
