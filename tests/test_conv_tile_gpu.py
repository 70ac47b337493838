"""The one-launch convolution at the edges of its tiles: pixel rectangles, channel chunks, output-channel tiles, borders."""
import numpy as np
import pytest

import oracle
from util import assert_parity, poison, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,Cin,H,W,Cout,KH,KW,s,p,d,act", [
    (1, 1, 1, 1, 1, 3, 3, 1, 1, 1, "none"),                # one output, all border
    (1, 3, 30, 29, 33, 7, 7, 4, 3, 1, "relu"),             # few channels in one chunk, channels off the 32-wide tile
    (2, 17, 13, 9, 65, 3, 3, 1, 1, 1, "none"),             # a last chunk of one channel
    (1, 64, 31, 33, 96, 3, 3, 2, 1, 1, "relu"),
    (1, 70, 8, 8, 32, 5, 5, 1, 2, 1, "none"),
    (1, 96, 40, 200, 64, 5, 5, 1, 2, 1, "none"),           # whole rounds of large tiles
    (1, 32, 12, 50, 160, 3, 1, (1, 2), (0, 1), (3, 1), "none"),
    (1, 16, 9, 300, 24, 1, 9, (2, 1), (4, 0), (1, 2), "none"),
    (4, 256, 15, 8, 256, 3, 3, 1, 1, 1, "relu"),           # long K, few pixels
    (1, 128, 64, 64, 256, 3, 3, 1, 1, 1, "none"),
    (1, 3, 260, 261, 144, 7, 7, 4, 3, 1, "none"),
    (1, 384, 5, 5, 384, 3, 3, 1, 0, 1, "none"),
    # strides that leave room for chunks of fewer than eight weights a channel, and a last chunk of one
    (1, 32, 512, 512, 84, 1, 1, (2, 8), 0, 1, "none"),
    (1, 33, 256, 300, 70, 1, 1, (8, 5), 0, 1, "relu"),
    (1, 35, 128, 100, 70, 3, 1, (8, 8), 0, 1, "none"),
    # the patch-gathering form: chunk pairs of several taps in a 64-deep tile, maps narrower than a piece, images past the CUs
    (1, 16, 70, 70, 64, 7, 7, 1, 3, 1, "none"),
    (1, 48, 65, 66, 72, 5, 5, (2, 1), (2, 0), (1, 2), "relu"),
    (1, 80, 37, 41, 130, 7, 7, 4, 3, 1, "none"),
    (2, 144, 30, 5, 256, 5, 3, 1, (1, 2), 1, "none"),      # seven columns with their borders
    (1, 192, 64, 3, 256, 3, 3, 1, (0, 1), 1, "relu"),      # one output column
    (2, 96, 120, 131, 96, 7, 7, 1, 3, 1, "none"),          # two workgroups a CU
    (3, 256, 33, 65, 64, 3, 3, 1, 1, (2, 1), "none"),
])
def test_conv_tiles(ctx, N, Cin, H, W, Cout, KH, KW, s, p, d, act):
    import torch
    import juliavision_amd as jv
    pair = lambda v: v if isinstance(v, tuple) else (v, v)
    s, p, d = pair(s), pair(p), pair(d)                    # (x, y)
    x = oracle.randn_f16((N, Cin, H, W), 1)
    w = oracle.randn_f16((Cout, Cin, KH, KW), 2, 0, 1.0 / np.sqrt(Cin * KH * KW))
    b = oracle.randn_f16((Cout,), 3, 0, 0.5)
    want = oracle.conv2d_f16(x, w, b, s[::-1], p[::-1], d[::-1], 1, act == "relu")
    out = poison(torch.empty(want.shape, dtype=torch.float16, device="cuda"))
    ctx.ws.reset()
    jv.convolution_(ctx, out, to_dev(x), to_dev(w), to_dev(b), s, p, d, 1, act=act)
    torch.cuda.synchronize()
    assert_parity(to_host(out), want, what=f"conv {Cin},{H},{W}->{Cout} k{KH}x{KW}")


@pytest.mark.parametrize("off", [1, 4])
@pytest.mark.parametrize("Cin,H,W,Cout,k,s,p", [
    (64, 32, 32, 64, 3, 1, 1), (256, 32, 32, 256, 3, 1, 1), (64, 24, 40, 48, 5, 1, 2), (128, 16, 24, 256, 1, 1, 0),      # extents of an implicit GEMM; 1 x 1
    (48, 30, 33, 64, 3, 2, 1), (96, 60, 57, 96, 5, 1, 2), (3, 70, 70, 40, 7, 4, 3), (70, 20, 20, 33, 3, 1, 1),           # patch copy, one launch, im2col
])
def test_operands_off_sixteen_bytes(ctx, Cin, H, W, Cout, k, s, p, off):
    """Weights sliced out of a flat buffer: every operand `off` elements behind an aligned address, guards around the result."""
    import torch
    import juliavision_amd as jv
    x, w = oracle.randn_f16((1, Cin, H, W), 1), oracle.randn_f16((Cout, Cin, k, k), 2, 0, 1.0 / np.sqrt(Cin * k * k))
    b = oracle.randn_f16((Cout,), 3, 0, 0.5)
    want = oracle.conv2d_f16(x, w, b, (s, s), (p, p), (1, 1), 1, False)

    def shifted(a):
        flat = torch.empty(a.size + off, dtype=torch.float16, device="cuda")
        flat[off:] = torch.from_numpy(a).cuda().reshape(-1)
        return flat[off:].view(a.shape)
    flat = torch.full((want.size + 2 * off,), float("nan"), dtype=torch.float16, device="cuda")
    out = flat[off:off + want.size].view(want.shape)
    ctx.ws.reset()
    jv.convolution_(ctx, out, shifted(x), shifted(w), shifted(b), (s, s), (p, p), (1, 1), 1)
    torch.cuda.synchronize()
    assert_parity(to_host(out), want, what=f"conv {Cin},{H},{W}->{Cout} k{k} off {off}")
    assert bool(torch.isnan(flat[:off]).all()) and bool(torch.isnan(flat[off + want.size:]).all())


@pytest.mark.parametrize("Cin,H,W,Cout,k", [
    (29, 64, 64, 32, 3), (30, 64, 64, 32, 3), (31, 40, 33, 70, 3), (31, 24, 24, 64, 2),      # staged as 32 channels
    (61, 20, 20, 32, 3), (62, 20, 20, 32, 3), (63, 20, 17, 33, 2),                           # as 64
    (29, 64, 5, 32, 3), (31, 40, 7, 40, 3), (62, 40, 5, 33, 2),                              # image rows shorter than a piece
])
def test_a_single_chunk_past_the_channels(ctx, Cin, H, W, Cout, k):
    """A chunk deeper than Cin: the weights that end inside a 16-byte piece, and the pieces behind them, which hold zeros whatever the tensor
    begins with (an infinity of channel 0 reaches channel 0's results alone)."""
    import ctypes as C

    import torch
    import juliavision_amd as jv
    from juliavision_amd import _lib as L
    p = k // 2
    assert L.CONV_KERNELS[L.load().mi_conv2d_f16_kernel(W, H, Cin, 1, k, k, Cout, 1, 1, p, p, 1, 1, 1, C.byref(C.c_size_t(0)))] == "tile"
    x, w, b = oracle.randn_f16((1, Cin, H, W), 1), oracle.randn_f16((Cout, Cin, k, k), 2, 0, 1.0 / np.sqrt(Cin * k * k)), oracle.randn_f16((Cout,), 3, 0, 0.5)
    outs = []
    for first in (w[0, 0, 0, 0], np.float16("inf")):
        w[0, 0, 0, 0] = first
        out = poison(torch.empty((1, Cout, H + 2 * p - k + 1, W + 2 * p - k + 1), dtype=torch.float16, device="cuda"))
        ctx.ws.reset()
        jv.convolution_(ctx, out, to_dev(x), to_dev(w), to_dev(b), (1, 1), (p, p), (1, 1), 1)
        torch.cuda.synchronize()
        if not outs:
            assert_parity(to_host(out), oracle.conv2d_f16(x, w, b, (1, 1), (p, p), (1, 1), 1, False), what=f"conv {Cin},{H},{W}->{Cout} k{k}")
        outs.append(to_host(out))
    assert np.array_equal(outs[0][:, 1:], outs[1][:, 1:])


@pytest.mark.parametrize("Cin", [3, 24])
@pytest.mark.parametrize("OW", [1, 2, 3, 5, 6, 7, 18, 37])
@pytest.mark.parametrize("Cout", [30, 33, 64])
def test_rows_that_end_between_four_pixels(ctx, Cin, OW, Cout):
    """Lanes exchange four pixels by four channels and store eight bytes: rows that end inside, channels that end inside, with a bias at an
    odd address and without, one chunk and several, nothing written past a row (the next one's first pixels follow it)."""
    import torch
    import juliavision_amd as jv
    H = 9
    x, w, b = oracle.randn_f16((2, Cin, H, OW), 1), oracle.randn_f16((Cout, Cin, 3, 3), 2, 0, 0.1), oracle.randn_f16((Cout + 1,), 3)
    held = torch.from_numpy(b).cuda()
    for bias in (held[1:], None):
        for act in ("none", "relu"):
            out = torch.full((2, Cout, H, OW), float("nan"), dtype=torch.float16, device="cuda")
            ctx.ws.reset()
            jv.convolution_(ctx, out, torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), bias, (1, 1), (1, 1), (1, 1), 1, act=act)
            want = oracle.conv2d_f16(x, w, None if bias is None else b[1:], (1, 1), (1, 1), (1, 1), 1, act == "relu")
            assert_parity(to_host(out), want, what=f"Cin{Cin} OW{OW} Cout{Cout} {act}")


@pytest.mark.parametrize("Cin,H,W,k", [(3, 20, 21, 3), (33, 20, 21, 3), (3, 20, 5, 3)])      # a chunk, several, by element
@pytest.mark.parametrize("Cout", [1, 2, 3, 4, 5, 7, 34, 61, 96, 98, 131])
def test_bias_of_every_channel(ctx, Cin, H, W, k, Cout):
    """Weights of zero: each channel is its bias, to the bit, where Cout ends inside four channels, inside a tile and inside four of them."""
    import torch
    import juliavision_amd as jv
    b = torch.arange(1, Cout + 2, dtype=torch.float16, device="cuda")
    out = torch.full((1, Cout, H, W), float("nan"), dtype=torch.float16, device="cuda")
    for bias in (b[1:], None):                             # at an odd address
        ctx.ws.reset()
        jv.convolution_(ctx, out, to_dev(oracle.randn_f16((1, Cin, H, W), 1)), torch.zeros((Cout, Cin, k, k), dtype=torch.float16, device="cuda"), bias,
                        (1, 1), (1, 1), (1, 1), 1)
        assert torch.equal(out, torch.zeros_like(out) if bias is None else bias.view(1, Cout, 1, 1).expand_as(out))


@pytest.mark.parametrize("N,Cin,H,W,Cout,KH,KW,s,p,d,act", [
    (1, 16, 60, 60, 96, 9, 9, 4, 4, 1, "relu"),            # eight taps a stage, more than a row of them
    (1, 32, 23, 17, 65, 5, 5, (2, 1), (2, 0), (1, 2), "none"),
    (2, 48, 13, 11, 96, 5, 3, 1, (1, 2), 1, "relu"),       # taps that end inside a stage, K inside its last one
    (1, 112, 10, 30, 70, 3, 3, 2, 1, 1, "none"),
    (1, 128, 8, 33, 32, 3, 3, 1, 1, 1, "none"),            # a tap a stage
    (1, 144, 31, 14, 144, 3, 3, 1, 1, 1, "none"),
    (3, 272, 7, 7, 31, 3, 3, 1, 1, 2, "relu"),             # channels and pixels off the tile
    (2, 192, 64, 3, 96, 3, 3, 1, (0, 1), 1, "none"),       # one output column
    (1, 256, 5, 5, 256, 3, 3, 1, 1, 1, "none"),
    (1, 384, 38, 11, 64, 7, 7, 4, 3, 1, "none"),           # two workgroups, 147 stages, four chains a wave
    (1, 272, 12, 26, 33, 1, 5, 1, (2, 0), 1, "none"),
    (1, 272, 26, 12, 33, 5, 1, 1, (0, 2), 1, "none"),      # one tap column
    (1, 256, 30, 112, 64, 3, 3, 1, 1, 1, "relu"),          # 210 workgroups
])
def test_patches_of_few_tiles(ctx, N, Cin, H, W, Cout, KH, KW, s, p, d, act):
    """The patch matrix in 32 x 32 tiles: taps and channels as the stages meet them.  Against 64 bits: products of fp16 values summed in
    fp32 leave 2^-24 a term of the sum of magnitudes (here below 3e-6 of the largest value), the result's own rounding 2^-11 of it."""
    import ctypes as C

    import torch
    import juliavision_amd as jv
    from juliavision_amd import _lib as L
    pair = lambda v: v if isinstance(v, tuple) else (v, v)
    s, p, d = pair(s), pair(p), pair(d)                    # (x, y)
    assert L.CONV_KERNELS[L.load().mi_conv2d_f16_kernel(W, H, Cin, N, KW, KH, Cout, *s, *p, *d, 1, C.byref(C.c_size_t(0)))] == "patch_gemm"
    assert L.GEMM_KERNELS[L.load().mi_conv2d_f16_patch_kernel(W, H, Cin, N, KW, KH, Cout, *s, *p, *d, 1)] == "deep"
    x, w = oracle.randn_f16((N, Cin, H, W), 1), oracle.randn_f16((Cout, Cin, KH, KW), 2, 0, 1.0 / np.sqrt(Cin * KH * KW))
    b = oracle.randn_f16((Cout,), 3, 0, 0.5)
    want = torch.nn.functional.conv2d(*(torch.from_numpy(a).double() for a in (x, w, b)), s[::-1], p[::-1], d[::-1]).numpy()
    if act == "relu":
        want = np.maximum(want, 0)
    assert -(-Cout // 32) * -(-want[0, 0].size // 32) * N <= 256
    out = poison(torch.empty(want.shape, dtype=torch.float16, device="cuda"))
    ctx.ws.reset()
    jv.convolution_(ctx, out, to_dev(x), to_dev(w), to_dev(b), s, p, d, 1, act=act)
    torch.cuda.synchronize()
    got = to_host(out).astype(np.float64)
    assert np.isfinite(got).all() and (np.abs(got - want) <= 2.0 ** -11 * np.abs(want) + 2.0 ** -24 + 3e-6 * np.abs(want).max()).all()
