"""J on the context's side stream beside K: the same J and K, bitwise, as one
stream gives, with new outputs on every call and eager work of the caller
between the calls."""

import pytest
import torch

from forte2_amd.jkbuilder import FockBuilder
from forte2_amd.workloads import orthonormal_C, synthetic_B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "bf16x3"])
@pytest.mark.parametrize("Q,N,noccs,xchunk", [(300, 96, [20], 0), (420, 130, [17, 13], 1 << 20), (2224, 384, [80], 0)])
def test_overlap_is_bitwise_the_same(dev, Q, N, noccs, xchunk, prec):
    print(f"[overlap] Q={Q} N={N} nocc={noccs} {prec}", flush=True)
    B = synthetic_B(Q, N, seed=N, device=dev)
    Cs = [orthonormal_C(N, o, seed=k, device=dev) for k, o in enumerate(noccs)]
    out = {}
    for overlap in (0, 1, -1):
        fb = FockBuilder(B=B, device=dev, precision=prec)
        fb.set_tuning("overlap_jk", overlap)
        if xchunk:
            fb.set_tuning("xchunk_bytes", xchunk)
        res = []
        for _ in range(3):
            J, K = fb.build_JK(Cs)
            res.append([x + 0.0 for x in J + K])  # the caller's own work right behind the build
            del J, K
        out[overlap] = res
    torch.cuda.synchronize()
    for overlap in (1, -1):
        for res in out[overlap]:
            assert all(torch.equal(a, b) for a, b in zip(res, out[0][0]))
