"""Masks that differ from query to query: both types, rows at any address, keys apart in memory, broadcast heads and batches, a tile
that the keys end in, lengths on top, rows with no key that counts."""
import numpy as np
import pytest

import oracle
from util import to_dev

pytestmark = pytest.mark.gpu


def _mask(kind, B, H, Lq, Lk, f32):
    import torch
    dt = torch.float32 if f32 else torch.float16
    m = to_dev(oracle.randn_f16((B, H, Lq, Lk), 7)).to(dt)
    if kind == "odd":                                     # every row at another odd address
        buf = torch.full((B, H, Lq, Lk + 3), float("nan"), dtype=dt, device="cuda").flatten()
        v = buf[1:1 + B * H * Lq * (Lk + 2)].view(B, H, Lq, Lk + 2)[..., :Lk]
        v.copy_(m)
        return v
    if kind == "keys_apart":
        return m.transpose(2, 3).contiguous().transpose(2, 3)
    if kind == "shared":                                  # one head's for all, as a position bias of the batch
        return m[:1, :1].contiguous().expand(B, H, Lq, Lk)
    m[..., Lk // 2:] = torch.where(torch.rand(m[..., Lk // 2:].shape, device="cuda") < 0.5, float("-inf"), m[..., Lk // 2:])
    m[:, :, ::5] = float("-inf")
    m[..., Lk - 1] = 0.5                                  # a key that counts in every row, in some the only one
    return m


@pytest.mark.parametrize("kind", ["odd", "keys_apart", "shared", "inf"])
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("B,H,Lq,Lk,E", [(2, 3, 2, 1, 64), (1, 2, 33, 31, 16), (2, 2, 63, 97, 32), (1, 2, 70, 333, 72), (2, 4, 130, 260, 64),
                                         (1, 3, 65, 545, 128), (3, 6, 200, 189, 16), (2, 20, 390, 391, 64), (1, 2, 40, 130, 40)])
def test_dense_masks(ctx, B, H, Lq, Lk, E, f32, kind):
    """Against 64 bits.  A call whose plan keeps fp32 is as near as fp32 sums leave it (4e-7, four times what a workgroup per row
    measures), the others within fp16 probabilities and queries' 6e-4."""
    import torch
    import juliavision_amd as jv
    q, k, v = (to_dev(oracle.randn_f16((B, H, L, E), s)) for s, L in ((1, Lq), (2, Lk), (3, Lk)))
    mask = _mask(kind, B, H, Lq, Lk, f32)
    lens = [Lk, Lk // 2 + 1, Lk][:B]
    out = torch.full((B, H, Lq, E), float("nan"), dtype=torch.float32, device="cuda")
    ctx.ws.reset()
    jv.sdpa(ctx, q, k, v, mask, kv_len=torch.tensor(lens, dtype=torch.int32, device="cuda") if kind == "odd" else None, out=out)
    s = torch.matmul(q.double().cpu(), k.double().cpu().transpose(2, 3)) / np.sqrt(E) + mask.double().cpu()
    if kind == "odd":
        for b, n in enumerate(lens):
            s[b, ..., n:] = float("-inf")
    want = torch.matmul(torch.softmax(s, -1), v.double().cpu())
    exact = type(jv.sdpaplan(ctx, q, k, v, mask)).__name__ == "RowsSDPAPlan" or (kind == "odd" and not f32) or (kind == "keys_apart" and Lk > 1)
    err = float((out.double().cpu() - want).norm() / want.norm())
    assert err <= (4e-7 if exact else 6e-4), (err, exact)
