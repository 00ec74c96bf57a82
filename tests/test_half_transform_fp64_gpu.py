"""The FP64 half-transform at the edges of its tiles: nbf below, at and past a
16-k step and odd (8-byte aligned rows), every column-block count class (one
and two row blocks per wave, one and two column tiles), a partial last row
tile, and an output row longer than the columns.

Tolerance: the rounding bound of a length-N sum, N eps |B| |C| per element.
"""

import pytest
import torch

from forte2_amd.jkbuilder import FockBuilder
from forte2_amd.workloads import synthetic_B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,N,ncol", [(1, 1, 1), (3, 15, 4), (5, 16, 16), (7, 17, 17), (20, 31, 31), (9, 33, 33), (600, 112, 70),
                                      (700, 130, 128), (40, 145, 144), (11, 161, 161), (6, 322, 320), (4, 340, 321)])
def test_half_transform(dev, Q, N, ncol):
    print(f"[half-transform] Q={Q} N={N} ncol={ncol}", flush=True)
    B = synthetic_B(Q, N, seed=N, device=dev)
    g = torch.Generator(device=dev)
    g.manual_seed(ncol)
    C = torch.randn((N, ncol), generator=g, device=dev, dtype=torch.float64)
    X = FockBuilder(B=B, device=dev).half_transform(C)
    ref = (B.cpu().reshape(-1, N) @ C.cpu()).reshape(Q, N, ncol)
    bound = N * 2.3e-16 * (B.abs().cpu().reshape(-1, N) @ C.abs().cpu()).reshape(Q, N, ncol) + 1e-300
    assert bool(((X.cpu() - ref).abs() <= 2 * bound).all())


@pytest.mark.parametrize("Q,N,n1,n2", [(1, 1, 1, 1), (5, 17, 3, 9), (5, 17, 9, 3), (20, 33, 16, 17), (7, 48, 48, 48), (300, 130, 21, 109),
                                       (300, 131, 110, 21), (6, 345, 325, 340), (6, 345, 340, 325), (4, 20, 45, 7)])
def test_mo_block(dev, Q, N, n1, n2):
    # either set first, one and two column tiles, a B that is not symmetric, a
    # column slice as C2, and more columns than functions in C1
    print(f"[mo-block] Q={Q} N={N} n1={n1} n2={n2}", flush=True)
    g = torch.Generator(device=dev)
    g.manual_seed(N + n1)
    B = torch.randn((Q, N, N), generator=g, device=dev, dtype=torch.float64)
    C1 = torch.randn((N, n1), generator=g, device=dev, dtype=torch.float64)
    C2 = torch.randn((N, n2 + 5), generator=g, device=dev, dtype=torch.float64)[:, 2:2 + n2]
    out = FockBuilder(B=B, device=dev).B_tensor_gen_block(C1, C2).cpu()
    b, c1, c2 = B.cpu(), C1.cpu(), C2.cpu()
    ref = torch.matmul(c1.T, b @ c2)
    bound = 2 * N * 2.3e-16 * torch.matmul(c1.abs().T, b.abs() @ c2.abs())
    assert bool(((out - ref).abs() <= 2 * bound).all())
