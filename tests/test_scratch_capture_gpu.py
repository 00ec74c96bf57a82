"""Limits of the no-alloc scratch array for K alone, and a captured build next
to an eager one on the same context."""

import ctypes

import pytest
import torch

from forte2_amd import _native as nat
from forte2_amd.workloads import orthonormal_C, synthetic_B

pytestmark = pytest.mark.gpu


def _ctx(dev, B):
    h = ctypes.c_void_p()
    nat.jk_check(nat.jk_lib().f2jk_ctx_create(dev.index, ctypes.byref(h)), "f2jk_ctx_create")
    nat.jk_check(nat.jk_lib().f2jk_set_B(h, nat.F2JK_F64, ctypes.c_void_p(B.data_ptr()), B.shape[0], B.shape[1]), "set_B")
    return h


class _Build:
    """One J/K (or K) build with its own outputs; ws None: the no-alloc entry."""

    def __init__(self, h, Cs, flags, ws):
        N = Cs[0].shape[0]
        self.h, self.flags, self.ws, self.Cs = h, flags, ws, Cs
        self.J = [torch.zeros(N, N, dtype=torch.float64, device=Cs[0].device) for _ in Cs]
        self.K = [torch.zeros_like(x) for x in self.J]
        self.args = (len(Cs), nat.ptr_array([C.data_ptr() for C in Cs]), nat.i64_array([C.shape[1] for C in Cs]),
                     nat.i64_array([C.stride(0) for C in Cs]), nat.ptr_array([x.data_ptr() for x in self.J]),
                     nat.ptr_array([x.data_ptr() for x in self.K]), nat.PREC["fp64"], flags)

    def __call__(self):
        lib, st = nat.jk_lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        if self.ws is None:
            rc = lib.f2jk_build_jk_noalloc(self.h, *self.args, st)
        else:
            rc = lib.f2jk_build_jk(self.h, *self.args, ctypes.c_void_p(self.ws.data_ptr()), self.ws.numel(), st)
        nat.jk_check(rc, "build")

    def out(self):
        return [x.clone() for x in self.J + self.K]


def _workspace(h, Cs, flags, dev):
    sz = ctypes.c_size_t()
    nocc = nat.i64_array([C.shape[1] for C in Cs])
    nat.jk_check(nat.jk_lib().f2jk_workspace_size(h, len(Cs), nocc, nat.PREC["fp64"], flags, ctypes.byref(sz)), "ws")
    return torch.empty(sz.value, dtype=torch.uint8, device=dev)


@pytest.mark.parametrize("N,o,nd", [(1233, 350, 3), (37, 11, 1)])
def test_k_alone_in_the_scratch_array(dev, N, o, nd):
    # (1233, 3 x 350): 12 N OPAD bytes of coefficients, 8 N OPAD of X at one P and
    # three N x N partials are 62 of the array's 67 MB
    print(f"[scratch] K alone N={N} nocc={nd}x{o}", flush=True)
    B = synthetic_B(3, N, seed=5, device=dev)
    Cs = [orthonormal_C(N, o, seed=k, device=dev) for k in range(nd)]
    h = _ctx(dev, B)
    b = _Build(h, Cs, nat.F2JK_WANT_K, None)
    b()
    torch.cuda.synchronize()
    for C, K in zip(Cs, b.K):
        ref = torch.zeros(N, N, dtype=torch.float64)
        for p in range(3):
            x = B[p].cpu() @ C.cpu()
            ref += x @ x.T
        assert (K.cpu() - ref).abs().max().item() <= 1e-10
    nat.jk_lib().f2jk_ctx_destroy(h)


def test_captured_build_beside_an_eager_one(dev):
    # J reads 158 MB: the eager build runs it on the context's side stream, which
    # must not have joined the capture
    N, Q = 256, 600
    print(f"[capture] N={N} Q={Q}", flush=True)
    B = synthetic_B(Q, N, seed=3, device=dev)
    C = orthonormal_C(N, 40, seed=1, device=dev)
    flags = nat.F2JK_WANT_J | nat.F2JK_WANT_K
    h = _ctx(dev, B)
    ws = _workspace(h, [C], flags, dev)
    eager, graphed = _Build(h, [C], flags, ws), _Build(h, [C], flags, None)
    eager(), graphed()
    torch.cuda.synchronize()
    ref_e, ref_g = eager.out(), graphed.out()
    other = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="relaxed"):
        graphed()
        with torch.cuda.stream(other):
            eager()
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(eager.out(), ref_e))
    for _ in range(3):
        for x in graphed.J + graphed.K:
            x.zero_()
        graph.replay()
        eager()  # eager work behind the replay
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(graphed.out(), ref_g))
        assert all(torch.equal(a, b) for a, b in zip(eager.out(), ref_e))
    nat.jk_lib().f2jk_ctx_destroy(h)
