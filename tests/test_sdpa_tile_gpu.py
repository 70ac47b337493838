"""flash_tile_kernel where it can go wrong: every head size it has, keys and queries around its 32-wide tiles, fewer tiles than
waves and more, a padding mask at either end of the keys, ragged lengths, values of one head beside the next."""
import numpy as np
import pytest

import oracle
from util import assert_parity, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mask", ["none", "right", "left", "len"])
@pytest.mark.parametrize("E", [16, 32, 64, 72, 128])
@pytest.mark.parametrize("B,H,Lq,Lk", [(1, 1, 2, 1), (2, 3, 31, 33), (2, 2, 65, 97), (1, 2, 33, 545), (3, 16, 520, 64), (12, 20, 90, 130)])
def test_tiles(ctx, B, H, Lq, Lk, E, mask):
    import torch
    import juliavision_amd as jv
    q, k, v = (oracle.randn_f16((B, L, 3, H, E), s, 0, 1.5) for s, L in ((1, Lq), (2, Lk), (3, Lk)))
    view = lambda a, i: torch.from_numpy(a).cuda()[:, :, i].transpose(1, 2)              # rows of 3 H E halves, read in place
    cut = [max(1, Lk - (7 * b + 40) % Lk) for b in range(B)]
    bias = np.zeros((B, 1, 1, Lk), np.float16)
    for b in range(B):
        if mask == "right":
            bias[b, ..., cut[b]:] = np.finfo(np.float16).min
        if mask == "left":
            bias[b, ..., :Lk - cut[b]] = -np.inf
    out = torch.full((B, Lq, H, E), float("nan"), dtype=torch.float16, device="cuda").transpose(1, 2)
    kv_len = torch.tensor(cut, dtype=torch.int32, device="cuda") if mask == "len" else None
    ctx.ws.reset()
    jv.sdpa(ctx, view(q, 0), view(k, 1), view(v, 2), to_dev(bias) if mask in ("right", "left") else None, kv_len=kv_len, out=out)
    torch.cuda.synchronize()
    dense = np.zeros((B, 1, 1, Lk), np.float32)
    for b in range(B):
        if mask in ("right", "len"):
            dense[b, ..., cut[b]:] = -np.inf
        if mask == "left":
            dense[b, ..., :Lk - cut[b]] = -np.inf
    s = np.einsum("bhqe,bhke->bhqk", *(np.float32(a[:, :, i]).transpose(0, 2, 1, 3) for a, i in ((q, 0), (k, 1)))) / np.sqrt(np.float32(E)) + dense
    p = np.exp(s - s.max(-1, keepdims=True))
    want = np.einsum("bhqk,bhke->bhqe", p / p.sum(-1, keepdims=True), np.float32(v[:, :, 2]).transpose(0, 2, 1, 3))
    assert_parity(to_host(out.contiguous()), want, what=f"{B}x{H} {Lq} over {Lk}, head size {E}, mask {mask}")


@pytest.mark.parametrize("garbage", [float("inf"), float("nan")])
@pytest.mark.parametrize("B,H,Lq,Lk,E", [(2, 3, 31, 97, 64), (3, 2, 5, 200, 72), (2, 8, 2, 64, 16), (2, 4, 40, 700, 128),          # few queries
                                         (3, 2, 70, 130, 32), (3, 4, 130, 300, 64), (2, 20, 400, 1500, 64), (2, 2, 100, 300, 96),     # every fused form
                                         (2, 16, 800, 1500, 64), (2, 1, 128, 8192, 64), (3, 2, 1, 300, 64), (3, 2, 1, 300, 80)])
def test_cache_slots_past_the_length_do_not_matter(ctx, B, H, Lq, Lk, E, garbage):
    """Keys at and past kv_len get weight exactly zero, whatever the unwritten slots of a caller's cache hold."""
    import torch
    import juliavision_amd as jv
    q, k, v = (to_dev(oracle.randn_f16((B, H, L, E), s)) for s, L in ((1, Lq), (2, Lk), (3, Lk)))
    lens = [Lk // 2 + 1, 1, Lk][:B]
    kv_len = torch.tensor(lens, dtype=torch.int32, device="cuda")
    outs = []
    for fill in (0.0, garbage):
        for b, n in enumerate(lens):
            k[b, :, n:], v[b, :, n:] = fill, fill
        out = torch.full((B, H, Lq, E), float("nan"), dtype=torch.float16, device="cuda")
        ctx.ws.reset()
        jv.sdpa(ctx, q, k, v, kv_len=kv_len, out=out)
        outs.append(out)
    assert bool(torch.isfinite(outs[0]).all()) and torch.equal(*outs)
