"""Extents at the edges of the GEMM kernels' tiles, ragged in every direction: K that ends inside a 64-deep tile, rows and columns
that are not multiples of eight halves, operands at odd addresses, few output tiles over a long K (K-groups)."""
import numpy as np
import pytest

import oracle
from util import assert_parity, to_dev, to_host

pytestmark = pytest.mark.gpu


def _check(ctx, T, K, F, layout, *, epi="none", residual=False, f32=False, shift=0, seed=1):
    import torch
    import juliavision_amd as jv
    X = oracle.randn_f16((T, K), seed, 0, 1.0 / np.sqrt(K))
    W = oracle.randn_f16((K, F), seed + 1)
    b = oracle.randn_f16((F,), seed + 2, 0, 0.02)
    R = oracle.randn_f16((T, F), seed + 3) if residual else None

    def place(a):                                         # `shift` elements into its allocation, guarded by NaNs on both sides
        buf = torch.full((a.size + shift + 64,), float("nan"), dtype=torch.float16, device="cuda")
        v = buf[shift:shift + a.size].view(a.shape)
        v.copy_(to_dev(a))
        return v
    w = place(W) if layout == "kf" else place(np.ascontiguousarray(W.T)).t()
    dt = torch.float32 if f32 else torch.float16
    pad = torch.full((T * F + shift + 64,), float("nan"), dtype=dt, device="cuda")
    out = pad[shift:shift + T * F].view(T, F)
    ctx.ws.reset()
    jv.matmul_(ctx, out, w, place(X), place(b), epi=epi, residual=None if R is None else _like(out, R))
    torch.cuda.synchronize()
    assert bool(torch.isnan(pad[:shift]).all()) and bool(torch.isnan(pad[shift + T * F:]).all()), "wrote outside the result"
    want = oracle.gemm_f16(X, W, b, epi=epi, residual=R)
    assert_parity(to_host(out), want, what=f"T{T} K{K} F{F} {layout}")


def _like(out, R):
    import torch
    r = torch.empty(out.numel() + 64, dtype=torch.float16, device="cuda")[:out.numel()].view(out.shape)
    r.copy_(to_dev(R))
    return r


@pytest.mark.parametrize("layout", ["kf", "fk"])
@pytest.mark.parametrize("T,K,F", [(64, 72, 64), (65, 120, 136), (129, 136, 200), (300, 1288, 512), (1544, 200, 1288), (2100, 328, 2056)])
def test_k_ends_inside_a_tile(ctx, T, K, F, layout):
    _check(ctx, T, K, F, layout, epi="gelu", residual=F != 200)


@pytest.mark.parametrize("layout", ["kf", "fk"])
@pytest.mark.parametrize("T,K,F", [(130, 1224, 104), (300, 1096, 264), (300, 136, 264), (2379, 72, 400), (454, 136, 4208), (839, 136, 4752), (1224, 200, 4888)])
def test_k_ends_inside_a_tile_of_every_size(ctx, T, K, F, layout):
    """The ring and every pipelined tile (64 x 64 to 128 x 256) with a K that is no multiple of 64."""
    _check(ctx, T, K, F, layout, residual=True)


@pytest.mark.parametrize("layout", ["kf", "fk"])
@pytest.mark.parametrize("T,K,F", [(1, 1, 1), (3, 7, 9), (2, 464, 73), (8, 9, 8), (17, 65, 33), (64, 63, 65), (70, 257, 129), (3, 2311, 106), (200, 311, 77),
                                   (1100, 130, 1999), (2049, 65, 2051), (33, 8, 24), (100, 64, 40)])
def test_ragged_in_every_direction(ctx, T, K, F, layout):
    _check(ctx, T, K, F, layout, residual=True)
    _check(ctx, T, K, F, layout, epi="relu", f32=True)


@pytest.mark.parametrize("layout", ["kf", "fk"])
@pytest.mark.parametrize("shift", [1, 4])
def test_odd_addresses(ctx, layout, shift):
    _check(ctx, 40, 192, 96, layout, shift=shift)
    _check(ctx, 5, 640, 64, layout, shift=shift, epi="gelu_tanh")


@pytest.mark.parametrize("N,Cin,H,W,Cout,KH,KW", [(1, 1, 1, 1, 1, 2, 2), (1, 65, 7, 9, 15, 2, 2), (2, 64, 8, 8, 16, 2, 2), (1, 130, 3, 43, 33, 2, 2),
                                                  (1, 8, 11, 13, 5, 3, 1), (2, 256, 96, 100, 64, 2, 2), (1, 72, 9, 5, 17, 3, 3)])
def test_upsampler_tiles(ctx, N, Cin, H, W, Cout, KH, KW):
    """Kernel == stride: pixels, channels and output channels off the 64-wide tiles, rows at odd addresses."""
    import torch
    import juliavision_amd as jv
    x, w = oracle.randn_f16((N, Cin, H, W), 1, 0, 0.5), oracle.randn_f16((Cin, Cout, KH, KW), 2, 0, 0.1)
    b = oracle.randn_f16((Cout,), 3, 0, 0.5)
    want = oracle.convtranspose2d_f16(x, w, b, (KH, KW))
    out = torch.full(want.shape, float("nan"), dtype=torch.float16, device="cuda")
    ctx.ws.reset()
    jv.convolutiontranspose_(ctx, out, to_dev(x), to_dev(w), to_dev(b), (KW, KH), (0, 0), (1, 1), (0, 0), 1)
    torch.cuda.synchronize()
    assert_parity(to_host(out), want, what="upsampler")
