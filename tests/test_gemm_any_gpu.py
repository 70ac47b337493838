"""The GEMM for operands of any extent and address: rows that end inside a sixteen-byte piece by every remainder, rows shorter than one,
one to five tiles of K and K-groups, a column tile that the rows end in."""
import numpy as np
import pytest

import oracle
from util import assert_parity, poison, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["kf", "fk"])
@pytest.mark.parametrize("T,K,F", [(70, 121 + r, 65 + r) for r in range(8)] + [(9, 3, 70), (9, 70, 3), (5, 7, 7), (130, 63, 9), (33, 65, 129), (40, 193, 17), (100, 5, 200), (100, 200, 5), (100, 5, 5),
                                                                                (70, 257, 71), (70, 321, 71), (17, 515, 614), (30, 1025, 77), (2200, 131, 2057)])
def test_every_remainder(ctx, T, K, F, layout):
    import torch
    import juliavision_amd as jv
    X, W, b = oracle.randn_f16((T, K), 1, 0, 1.0 / np.sqrt(K)), oracle.randn_f16((K, F), 2), oracle.randn_f16((F,), 3, 0, 0.02)

    def place(a):                                         # an odd address, NaNs on both sides: nothing outside a row may count
        buf = torch.full((a.size + 65,), float("nan"), dtype=torch.float16, device="cuda")
        v = buf[1:1 + a.size].view(a.shape)
        v.copy_(to_dev(a))
        return v
    out = poison(torch.empty((T, F), dtype=torch.float16, device="cuda"))
    ctx.ws.reset()
    jv.matmul_(ctx, out, place(W) if layout == "kf" else place(np.ascontiguousarray(W.T)).t(), place(X), place(b))
    torch.cuda.synchronize()
    assert_parity(to_host(out), oracle.gemm_f16(X, W, b), what=f"T{T} K{K} F{F} {layout}")
