"""Blocks of P of the MO-basis transform: wide sets take enough P per block for
a round of workgroups in both launches, and the result is that of torch."""

import ctypes

import pytest
import torch

from forte2_amd import _native as nat
from forte2_amd.jkbuilder import FockBuilder
from forte2_amd.workloads import orthonormal_C, synthetic_B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("naux,nbf,n1,n2,least", [(1800, 640, 128, 128, 500), (1800, 640, 320, 320, 100),
                                                  (1800, 640, 640, 640, 25), (1500, 499, 99, 99, 500)])
def test_block_fills_the_chip(dev, naux, nbf, n1, n2, least):
    # no kernel runs: B is registered by its shape.  `least`: P of a block of 512
    # workgroups (1, 5, 20 and 0.9 per P in the smaller launch)
    print(f"[mo-plan] naux={naux} nbf={nbf} n={n1},{n2}", flush=True)
    lib, h, size = nat.jk_lib(), ctypes.c_void_p(), ctypes.c_size_t()
    nat.jk_check(lib.f2jk_ctx_create(dev.index, ctypes.byref(h)), "create")
    B = torch.empty(256, dtype=torch.float64, device=dev)
    nat.jk_check(lib.f2jk_set_B(h, nat.F2JK_F64, ctypes.c_void_p(B.data_ptr()), naux, nbf), "set_B")
    nat.jk_check(lib.f2jk_mo_block_workspace_size(h, n1, n2, ctypes.byref(size)), "size")
    per_p = 8 * nbf * min(n1, n2)
    assert least * per_p <= size.value <= (512 << 20) + 8 * (nbf + 32) * (n1 + n2 + 64)
    lib.f2jk_ctx_destroy(h)


@pytest.mark.parametrize("Q,N,n1,n2", [(700, 340, 200, 200), (331, 340, 330, 190), (500, 301, 70, 300)])
def test_blocks(dev, Q, N, n1, n2):
    print(f"[mo-plan] Q={Q} N={N} n={n1},{n2}", flush=True)
    B = synthetic_B(Q, N, seed=N, device=dev)
    C1, C2 = orthonormal_C(N, n1, seed=1, device=dev), orthonormal_C(N, n2, seed=2, device=dev)
    out = FockBuilder(B=B, device=dev, j_sparse=False).B_tensor_gen_block(C1, C2)
    ref = torch.matmul(C1.T.contiguous(), torch.matmul(B, C2))
    # two FP64 sums of at most 340 terms of order 0.05
    assert float((out - ref).abs().max()) <= 1e-12
