"""The 256-row BF16x3 half-transform at odd tile widths and with a partial last
column tile: K bitwise as with the 128-row kernel, which runs the same products
in the same order, and within the split bound of FP64."""

import pytest
import torch

from forte2_amd.jkbuilder import FockBuilder
from forte2_amd.workloads import orthonormal_C, synthetic_B

pytestmark = pytest.mark.gpu


# occupied units of 32 columns: 5, 7, 9 (one tile of 10), 11 (2 x 6), 13 (2 x 7), 17 (3 x 6)
@pytest.mark.parametrize("Q,N,noccs", [(60, 200, [150]), (40, 260, [110, 105]), (30, 300, [270]), (33, 340, [330]),
                                       (20, 420, [410]), (9, 544, [540])])
def test_widths(dev, Q, N, noccs):
    print(f"[tall] Q={Q} N={N} nocc={noccs}", flush=True)
    B = synthetic_B(Q, N, seed=N, device=dev)
    Cs = [orthonormal_C(N, o, seed=k, device=dev) for k, o in enumerate(noccs)]
    out = {}
    for rows in (128, 256):
        fb = FockBuilder(B=B, device=dev, precision="bf16x3")
        fb.set_tuning("kx_rows", rows)
        fb.set_tuning("bf16_nbw_max", 10)
        out[rows] = fb.build_K(Cs)
        fb.release()
    for C, a, b in zip(Cs, out[128], out[256]):
        x = torch.matmul(B, C).transpose(0, 1).reshape(N, -1)
        ref = x @ x.T
        assert torch.equal(a, b)
        assert float((b - ref).abs().max()) <= 2e-5 * float(ref.abs().max())
