"""What a caller's workspace has to hold (no kernel runs; B is registered by
its shape, never read): the size of a J and K build is enough for J and for K
alone with the same arguments, and the row sums kept beside X do not split a
job whose X fits its chunk."""

import ctypes

import pytest
import torch

from forte2_amd import _native as nat

pytestmark = pytest.mark.gpu

J, K = nat.F2JK_WANT_J, nat.F2JK_WANT_K


def _ctx(dev, naux, nbf, xchunk=0):
    lib, h = nat.jk_lib(), ctypes.c_void_p()
    nat.jk_check(lib.f2jk_ctx_create(dev.index, ctypes.byref(h)), "create")
    B = torch.empty(256, dtype=torch.float64, device=dev)
    nat.jk_check(lib.f2jk_set_B(h, nat.F2JK_F64, ctypes.c_void_p(B.data_ptr()), naux, nbf), "set_B")
    if xchunk:
        nat.jk_check(lib.f2jk_set_tuning(h, b"xchunk_bytes", xchunk), "xchunk")
    return h, B


@pytest.mark.parametrize("naux,nbf,noccs,xchunk", [(9414, 1412, [68], 0), (7430, 1478, [46], 0), (3932, 945, [282], 0),
                                                   (940, 144, [14, 14], 1 << 20), (834, 118, [19, 19], 1 << 21),
                                                   (7456, 1493, [375] * 4, 1 << 22), (139, 24, [5], 0)])
def test_jk_size_covers_j_and_k_alone(dev, naux, nbf, noccs, xchunk):
    print(f"[plans] naux={naux} nbf={nbf} nocc={noccs} xchunk={xchunk}", flush=True)
    lib = nat.jk_lib()
    h, B = _ctx(dev, naux, nbf, xchunk)
    nd, nocc = len(noccs), nat.i64_array(noccs)

    def size(n, flags):
        b = ctypes.c_size_t()
        nat.jk_check(lib.f2jk_workspace_size(h, nd, n, nat.PREC["fp64"], flags, ctypes.byref(b)), "size")
        return b.value

    jk = size(nocc, J | K)
    assert jk >= size(nocc, K)
    assert jk >= size(nocc, J)   # J from C
    assert jk >= size(None, J)   # J from D
    lib.f2jk_ctx_destroy(h)


@pytest.mark.parametrize("naux,nbf,nocc", [(6700, 1000, 80), (7430, 1478, 46)])
def test_grouped_job_at_the_chunk_limit(dev, naux, nbf, nocc):
    # X of the first is 4.288 GB, the chunk 4.295 GB
    lib = nat.jk_lib()
    h, B = _ctx(dev, naux, nbf)
    size = (ctypes.c_size_t * 1)()
    rc = lib.f2jk_group_workspace_size(nat.ptr_array([h.value]), 1, (ctypes.c_int * 1)(1), nat.i64_array([nocc]),
                                       nat.PREC["fp64"], J | K, size)
    assert rc == 0 and size[0] > 8 * naux * nbf * nocc
    lib.f2jk_ctx_destroy(h)
