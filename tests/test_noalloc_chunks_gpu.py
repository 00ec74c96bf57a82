"""Chunks of X in the no-alloc scratch array: where J's share of the array makes
a chunk miss it by little, the chunk is cut by that and not in half."""

import ctypes

import pytest
import torch

from forte2_amd import _native as nat
from forte2_amd.workloads import orthonormal_C, synthetic_B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,N,o", [(2224, 384, 76)])
def test_j_does_not_double_the_chunks(dev, Q, N, o):
    print(f"[no-alloc chunks] Q={Q} N={N} nocc={o}", flush=True)
    lib, h = nat.jk_lib(), ctypes.c_void_p()
    B = synthetic_B(Q, N, seed=1, device=dev)
    C = orthonormal_C(N, o, seed=2, device=dev)
    J, K = (torch.empty((N, N), dtype=torch.float64, device=dev) for _ in range(2))
    nat.jk_check(lib.f2jk_ctx_create(dev.index, ctypes.byref(h)), "create")
    nat.jk_check(lib.f2jk_set_B(h, nat.F2JK_F64, ctypes.c_void_p(B.data_ptr()), Q, N), "set_B")
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    chunks = {}
    for flags in (nat.F2JK_WANT_K, nat.F2JK_WANT_J | nat.F2JK_WANT_K):
        nat.jk_check(lib.f2jk_build_jk_noalloc(h, 1, nat.ptr_array([C.data_ptr()]), nat.i64_array([o]), nat.i64_array([o]),
                                               nat.ptr_array([J.data_ptr()]), nat.ptr_array([K.data_ptr()]),
                                               nat.PREC["fp64"], flags | nat.F2JK_TIMING, st), "build")
        torch.cuda.synchronize()
        n = (ctypes.c_int * len(nat.PHASES))()
        nat.jk_check(lib.f2jk_last_launches(h, n, len(nat.PHASES)), "launches")
        chunks[flags] = n[nat.PHASES.index("kx")]
        x = torch.matmul(B, C).transpose(0, 1).reshape(N, -1)
        assert float((K - x @ x.T).abs().max()) <= 1e-10
    # J takes 7 of the array's 67 MB
    assert chunks[nat.F2JK_WANT_J | nat.F2JK_WANT_K] <= 1.5 * chunks[nat.F2JK_WANT_K]
    lib.f2jk_ctx_destroy(h)
