"""flash_tile_kernel where it can go wrong: every head size it has, keys and queries around its 32-wide tiles, fewer tiles than
waves and more, a padding mask at either end of the keys, ragged lengths, values of one head beside the next."""
import numpy as np
import pytest

import oracle
from util import assert_parity, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mask", ["none", "right", "left", "len"])
@pytest.mark.parametrize("E", [16, 32, 64, 72, 128])
@pytest.mark.parametrize("B,H,Lq,Lk", [(1, 1, 2, 1), (2, 3, 31, 33), (2, 2, 65, 97), (1, 2, 33, 545), (3, 16, 520, 64), (12, 20, 90, 130), (6, 20, 159, 159)])
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


@pytest.mark.parametrize("fill", [-65504.0, -1000.0, -np.inf])
@pytest.mark.parametrize("kind", ["key16", "dense16", "dense32"])
@pytest.mark.parametrize("B,H,Lq,Lk,E", [(1, 2, 100, 300, 64), (2, 3, 20, 300, 64), (1, 2, 70, 330, 72), (1, 2, 33, 300, 16), (1, 2, 65, 260, 128),
                                         (2, 2, 90, 300, 40), (1, 3, 130, 270, 80), (1, 2, 70, 270, 120), (2, 16, 830, 1400, 64), (2, 16, 300, 520, 64)])
def test_left_padding(ctx, B, H, Lq, Lk, E, kind, fill):
    """Keys masked from the left, by more than a tile or block of them, in every form that carries a mask: a reference point that
    followed the masked keys down would cost the first keys that count their last bits (fp32 steps of 2^-7 at -65504 log2(e)) or
    every number (0 x infinity).  With fp16 probabilities and queries such a result is within 4e-4 of fp64; rows whose keys are
    all masked by one finite value are the softmax of their scores, to the steps that fp32 leaves of s - 65504."""
    import torch
    import juliavision_amd as jv
    q, k, v = (to_dev(oracle.randn_f16((B, H, L, E), s)) for s, L in ((1, Lq), (2, Lk), (3, Lk)))
    pad = [Lk // 3 + 77, 40][:B]
    mask = torch.zeros((B, 1, 1 if kind == "key16" else Lq, Lk), dtype=torch.float32 if kind == "dense32" else torch.float16, device="cuda")
    for b, n in enumerate(pad):
        mask[b, ..., :n] = fill
    whole = kind != "key16" and fill != -np.inf
    if whole:
        mask[:, :, ::7] = fill                                                        # rows without a key that counts
    out = torch.full((B, H, Lq, E), float("nan"), dtype=torch.float32, device="cuda")
    ctx.ws.reset()
    jv.sdpa(ctx, q, k, v, mask, out=out)
    s = torch.matmul(q.double().cpu(), k.double().cpu().transpose(2, 3)) / np.sqrt(E) + mask.double().cpu()
    want, got = torch.matmul(torch.softmax(s, -1), v.double().cpu()), out.double().cpu()
    rel = lambda a, b: float((a - b).norm() / b.norm())
    some = torch.ones(Lq, dtype=torch.bool)
    if whole:
        some[::7] = False
        assert rel(got[:, :, ~some], want[:, :, ~some]) <= 1e-2
    assert rel(got[:, :, some], want[:, :, some]) <= 6e-4


@pytest.mark.parametrize("B,H,Lq,Lk,E", [(1, 2, 100, 300, 64), (2, 20, 1500, 1500, 64), (1, 2, 130, 270, 80), (1, 2, 70, 270, 120), (1, 2, 40, 300, 64)])
def test_scores_far_below_zero(ctx, B, H, Lq, Lk, E):
    """Every score near -200: the first block settles the reference point there, with nothing to rescale yet."""
    import torch
    import juliavision_amd as jv
    c = 2.0 ** round(np.log2(np.sqrt(200 / np.sqrt(E))))                              # exact in fp16: all queries round alike
    q = torch.full((B, H, Lq, E), c, dtype=torch.float16, device="cuda")
    k, v = -q.new_full((B, H, Lk, E), c), to_dev(oracle.randn_f16((B, H, Lk, E), 3))
    out = torch.full((B, H, Lq, E), float("nan"), dtype=torch.float16, device="cuda")
    ctx.ws.reset()
    jv.sdpa(ctx, q, k, v, out=out)
    want = v.float().mean(2, keepdim=True).expand(out.shape)                          # equal scores: equal weights
    assert float((out.float() - want).norm() / want.norm()) <= 1e-2


# Relative errors (2-norm, fp32 result) against fp64 of a workgroup per query row, which keeps everything in fp32 and answered these
# calls before there were tiles: measured on these operands, the third digit rounded up.
@pytest.mark.parametrize("B,H,Lq,Lk,E,mask,rows", [
    (8, 8, 32, 32, 64, False, 1.18e-7), (2, 8, 23, 300, 64, True, 1.44e-7), (4, 20, 60, 1500, 64, True, 1.91e-7), (16, 8, 40, 256, 64, False, 1.46e-7),
    (8, 16, 2, 1000, 64, False, 1.66e-7), (2, 8, 23, 300, 16, True, 1.44e-7), (4, 20, 60, 1500, 16, True, 1.98e-7), (16, 8, 40, 256, 32, False, 1.62e-7),
    (2, 8, 23, 300, 128, False, 1.66e-7), (8, 16, 2, 1000, 128, True, 1.79e-7)])
def test_few_queries_keep_fp32(ctx, B, H, Lq, Lk, E, mask, rows):
    import torch
    import juliavision_amd as jv
    gen = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = (torch.randn(B, H, L, E, generator=gen, device="cuda").half() for L in (Lq, Lk, Lk))
    bias = None
    if mask:
        length = Lk - torch.randint(0, Lk // 3, (B, 1), generator=gen, device="cuda")
        bias = torch.where(torch.arange(Lk, device="cuda")[None] < length, 0.0, -65504.0).half().view(B, 1, 1, Lk)
    plan = jv.sdpaplan(ctx, q, k, v, bias)
    assert type(plan).__name__ == "RowsSDPAPlan" and plan.kernel == "tiles_f32", plan
    out = torch.full((B, H, Lq, E), float("nan"), dtype=torch.float32, device="cuda")
    ctx.ws.reset()
    jv.sdpa(ctx, q, k, v, bias, out=out)
    s = torch.matmul(q.double().cpu(), k.double().cpu().transpose(2, 3)) / np.sqrt(E) + (0.0 if bias is None else bias.double().cpu())
    want = torch.matmul(torch.softmax(s, -1), v.double().cpu())
    assert float((out.double().cpu() - want).norm() / want.norm()) <= rows


@pytest.mark.parametrize("B,H,Lq,Lk,E,mask,kernel", [(1, 4, 7, 64, 64, False, "rows"), (1, 20, 1, 448, 64, False, "one_query"), (1, 8, 23, 700, 16, False, "tiles"),
                                                     (1, 8, 23, 4096, 16, False, "fused"), (1, 16, 4096, 4096, 64, False, "fused"), (1, 6, 1370, 1370, 64, True, "tiles"),
                                                     (2, 8, 23, 300, 72, True, "tiles_f32")])
def test_the_plan_names_the_kernel(ctx, B, H, Lq, Lk, E, mask, kernel):
    import torch
    import juliavision_amd as jv
    q, k, v = (torch.zeros(B, H, L, E, dtype=torch.float16, device="cuda") for L in (Lq, Lk, Lk))
    assert jv.sdpaplan(ctx, q, k, v, q.new_zeros(B, 1, 1, Lk) if mask else None).kernel == kernel


@pytest.mark.parametrize("B", [11, 24])
@pytest.mark.parametrize("mask", [False, True])
@pytest.mark.parametrize("Lk", [31, 70, 160])
def test_grids_around_the_waves_that_fit(ctx, B, mask, Lk):
    """Heads of 64 read V ahead of the exponentials while all waves of the grid fit the registers that takes (880 workgroups of two to four
    waves here, and 1920), behind them past that.  Probabilities are rounded to fp16 (2^-11 of the result at most), the result once more."""
    import torch
    import juliavision_amd as jv
    q, k, v = (to_dev(oracle.randn_f16((B, 16, L, 64), s, 0, 1.5)) for s, L in ((1, 160), (2, Lk), (3, Lk)))
    bias = torch.zeros((B, 1, 1, Lk), dtype=torch.float16, device="cuda")
    for b in range(B if mask else 0):
        bias[b, ..., Lk - b % Lk:] = torch.finfo(torch.float16).min
    out = torch.full((B, 16, 160, 64), float("nan"), dtype=torch.float16, device="cuda")
    ctx.ws.reset()
    jv.sdpa(ctx, q, k, v, bias if mask else None, None, out=out)
    s = torch.matmul(q.float(), k.float().transpose(2, 3).contiguous()) / 8.0 + bias.float()
    want = torch.matmul(torch.softmax(s, -1), v.float())
    assert ((out.float() - want).norm() / want.norm()).item() <= 2.0 ** -10
    assert_parity(to_host(out), want.cpu().numpy(), what=f"{B} x 16 heads, {Lk} keys")
