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


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("E,half", [(16, False), (32, False), (64, False), (72, True), (128, False)])
@pytest.mark.parametrize("Lq,apart", [(63, False), (130, True)])
def test_rows_without_a_key(ctx, Lq, apart, E, half, f32):
    """Rows of -inf give zeros, beside rows of the same 32-query tile that have keys.  fp16 results bring head size 72 here too."""
    import torch
    import juliavision_amd as jv
    B, H, Lk = 2, 3, 189
    q, k, v = (to_dev(oracle.randn_f16((B, H, L, E), s)) for s, L in ((1, Lq), (2, Lk), (3, Lk)))
    mask = to_dev(oracle.randn_f16((B, H, Lq, Lk), 7)).to(torch.float32 if f32 else torch.float16)
    mask[:, :, 1::3] = float("-inf")
    mask[0, 1] = float("-inf")                            # whole tiles of them
    mask[:, :, ::3, 40:] = float("-inf")                  # and rows whose keys are the first wave's
    if apart:
        mask = mask.transpose(2, 3).contiguous().transpose(2, 3)
    out = torch.full((B, H, Lq, E), float("nan"), dtype=torch.float16 if half else torch.float32, device="cuda")
    ctx.ws.reset()
    jv.sdpa(ctx, q, k, v, mask, out=out)
    s = torch.matmul(q.double().cpu(), k.double().cpu().transpose(2, 3)) / np.sqrt(E) + mask.double().cpu()
    want = torch.matmul(torch.softmax(s, -1), v.double().cpu()).nan_to_num(0.0)
    got, dead = out.double().cpu(), torch.isneginf(mask.cpu()).all(-1)
    assert dead.any() and bool((got[dead] == 0).all())
    # fp32 sums and products of an fp16 pair each: as test_dense_masks
    assert float((got - want).norm() / want.norm()) <= (2.0 ** -11 if half else 4e-7)


@pytest.mark.parametrize("fill", [-1e4, -1e7, -1e9, -1e30, "min"])
@pytest.mark.parametrize("apart", [False, True])
@pytest.mark.parametrize("E,half", [(16, False), (32, False), (64, False), (72, True), (128, False)])
def test_large_finite_masks(ctx, E, half, apart, fill):
    """fp32 masks that exclude keys by a large finite number: padding in front, behind, on both sides, none, and rows masked
    throughout.  Scores have a standard deviation of 3.  A key that counts outweighs the others without trace; a row without
    one is its scores rounded to the mask's spacing, which from 1e9 on is one value: the mean of V (below, such rows are left out)."""
    import torch
    import juliavision_amd as jv
    B, H, Lq, Lk = 1, 2, 63 if not apart else 130, 545
    lowest = float(np.finfo(np.float32).min) if fill == "min" else fill
    q, k, v = (to_dev(oracle.randn_f16((B, H, L, E), s)) for s, L in ((11, Lq), (12, Lk), (13, Lk)))
    q = (q.float() * 3).half()
    m = torch.zeros((B, H, Lq, Lk), dtype=torch.float32)
    for i in range(Lq):
        front, behind = ((300, 0), (0, 412), (100, 130), (0, 0), (544, 0), (0, 544))[i % 6]
        m[:, :, i, :front] = lowest
        m[:, :, i, Lk - behind:] = lowest
    if lowest <= -1e9:
        m[:, :, 7::9] = lowest
    mask = m.cuda()
    if apart:
        mask = mask.transpose(2, 3).contiguous().transpose(2, 3)
    out = torch.full((B, H, Lq, E), float("nan"), dtype=torch.float16 if half else torch.float32, device="cuda")
    ctx.ws.reset()
    jv.sdpa(ctx, q, k, v, mask, out=out)
    s = (torch.matmul(q.double().cpu(), k.double().cpu().transpose(2, 3)) / np.sqrt(E) + m.double()).float().double()
    want = torch.matmul(torch.softmax(s, -1), v.double().cpu())
    assert bool(torch.isfinite(out).all())
    err = (out.double().cpu() - want).norm(dim=-1) / want.norm(dim=-1)
    # per row: eight roundings of scores of up to 20 (2^-21 each) with fp32 results, half a unit of fp16 with fp16 ones
    assert float(err.max()) <= (2.0 ** -10 if half else 4e-6), float(err.max())
