"""Five to eight rows against [F][K] weights, on the matrix cores: K that ends inside a 32-deep step and a wave's share, one step and
many, columns off the tiles of eight and sixteen, the norm in front bit for bit as its own launch."""
import numpy as np
import pytest

import oracle
from util import assert_parity, poison, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [5, 8])
@pytest.mark.parametrize("K,F", [(8, 16), (24, 3), (40, 7), (256, 130), (264, 17), (1280, 33), (1288, 2100), (2568, 24), (5128, 40), (8192, 9)])
def test_rows(ctx, T, K, F):
    import torch
    import juliavision_amd as jv
    X, W, b = oracle.randn_f16((T, K), 1, 0, 1.0 / np.sqrt(K)), oracle.randn_f16((K, F), 2), oracle.randn_f16((F,), 3, 0, 0.02)
    R, g, beta = oracle.randn_f16((T, F), 4), oracle.randn_f16((K,), 5, 1.0, 0.1), oracle.randn_f16((K,), 6, 0, 0.1)
    w, dx, db = to_dev(np.ascontiguousarray(W.T)).t(), to_dev(X), to_dev(b)
    new = lambda dt=torch.float16: poison(torch.empty((T, F), dtype=dt, device="cuda"))
    for epi, res, dt in (("gelu", None, torch.float16), ("none", R, torch.float16), ("relu", None, torch.float32)):
        out = new(dt)
        ctx.ws.reset()
        jv.matmul_(ctx, out, w, dx, db, epi=epi, residual=None if res is None else to_dev(res))
        assert_parity(to_host(out), oracle.gemm_f16(X, W, b, epi=epi, residual=res), what=f"T{T} K{K} F{F} {epi}")
    # fp32 results: sums of K products in fp32, each half exact (2^-24 sqrt(K) of a result that is a sum of as many, with room)
    exact = X.astype(np.float64) @ W.astype(np.float64) + b.astype(np.float64)
    out = new(torch.float32)
    ctx.ws.reset()
    jv.matmul_(ctx, out, w, dx, db)
    assert np.linalg.norm(to_host(out) - exact) <= 2.0 ** -24 * max(8.0, np.sqrt(K)) * np.linalg.norm(exact)
    h, folded, apart = torch.empty((T, K), dtype=torch.float16, device="cuda"), new(), new()
    ctx.ws.reset()
    jv.ln_matmul_(ctx, folded, w, dx, to_dev(g), to_dev(beta), 1e-5, db)
    jv.layernorm_(ctx, h, None, None, dx, to_dev(g), to_dev(beta), K, 1e-5)
    ctx.ws.reset()
    jv.matmul_(ctx, apart, w, h, db)
    if K <= 4096:                                         # the norm kernel walks longer rows in another order
        assert torch.equal(folded, apart)


@pytest.mark.parametrize("beta", [False, True])
@pytest.mark.parametrize("K", [8, 40, 1280, 1288])
def test_norm_without_gamma_of_rows_far_from_zero(ctx, K, beta):
    """The columns that pad a wave's share have no value to normalise: minus the mean times 1 / sigma is beyond fp16 here."""
    import torch
    import juliavision_amd as jv
    T, F = 6, 40
    X = np.full((T, K), 900.0, np.float16)
    X[1::2, ::3] = 901.0
    W, be = oracle.randn_f16((K, F), 2, 0, 1.0 / np.sqrt(K)), oracle.randn_f16((K,), 6, 0, 0.1)
    out = poison(torch.empty((T, F), dtype=torch.float16, device="cuda"))
    ctx.ws.reset()
    jv.ln_matmul_(ctx, out, to_dev(np.ascontiguousarray(W.T)).t(), to_dev(X), None, to_dev(be) if beta else None, 1e-5, None)
    h = poison(torch.empty((T, K), dtype=torch.float16, device="cuda"))
    jv.layernorm_(ctx, h, None, None, to_dev(X), None, to_dev(be) if beta else None, K, 1e-5)
    assert_parity(to_host(out), oracle.gemm_f16(to_host(h), W), what=f"K{K} beta {beta}")


@pytest.mark.parametrize("T", [1, 2, 3, 4, 6, 8])
@pytest.mark.parametrize("K,F", [(8, 12353), (512, 2053), (520, 8197), (1024, 3071), (1032, 4099), (1288, 5117), (1536, 16397), (3072, 37), (4104, 21), (6152, 19)])
def test_rows_of_every_depth_and_width(ctx, T, K, F):
    """The kernels are picked by K (chunks asked for at the top) and F (columns a wave, workgroups that walk): either side of each edge,
    columns off every group, with a bias and without, with the norm in front and without."""
    import torch
    import juliavision_amd as jv
    X, W, b = oracle.randn_f16((T, K), 1, 0, 1.0), oracle.randn_f16((K, F), 2, 0, 1.0 / np.sqrt(K)), oracle.randn_f16((F,), 3, 0, 0.1)
    R, g, beta = oracle.randn_f16((T, F), 4), oracle.randn_f16((K,), 5, 1.0, 0.1), oracle.randn_f16((K,), 6, 0, 0.1)
    w, dx, db, dr = to_dev(np.ascontiguousarray(W.T)).t(), to_dev(X), to_dev(b), to_dev(R)
    new = lambda: poison(torch.empty((T, F), dtype=torch.float16, device="cuda"))
    h = torch.empty((T, K), dtype=torch.float16, device="cuda")
    jv.layernorm_(ctx, h, None, None, dx, to_dev(g), to_dev(beta), K, 1e-5)
    for bias, res in ((db, dr), (None, None)):
        plain, folded, apart = new(), new(), new()
        kw = {"residual": res, "epi": "gelu"}
        ctx.ws.reset()
        jv.matmul_(ctx, plain, w, dx, bias, **kw)
        assert_parity(to_host(plain), oracle.gemm_f16(X, W, None if bias is None else b, epi="gelu", residual=None if res is None else R), what=f"T{T} K{K} F{F}")
        ctx.ws.reset()
        jv.ln_matmul_(ctx, folded, w, dx, to_dev(g), to_dev(beta), 1e-5, bias, **kw)
        ctx.ws.reset()
        jv.matmul_(ctx, apart, w, h, bias, **kw)
        if K <= 4096:                                     # the norm kernel walks longer rows in another order
            assert torch.equal(folded, apart)
        else:
            assert_parity(to_host(folded), to_host(apart), what=f"norm T{T} K{K} F{F}")


@pytest.mark.parametrize("T", [1, 2, 3, 8])
@pytest.mark.parametrize("K,F", [(8, 64), (64, 24), (72, 8192), (128, 8200), (136, 8), (512, 40), (768, 136), (776, 264), (1280, 72), (1280, 5120), (1288, 64)])
def test_rows_against_kf_weights(ctx, T, K, F):
    """[K][F] weights at the ends of the range that runs as 32 x 32 tiles: K of part of a stage, of one and of ten, one column tile and 256 of
    them; one past each end as slices of K.  The rows lie apart in memory.  Error as in test_rows; the norm in front has the bits of the two calls."""
    import ctypes as C

    import torch
    import juliavision_amd as jv
    from juliavision_amd import _lib as L
    slices = C.c_int(0)
    ctx.lib.mi_gemm_f16_plan_caps(None, 0x10000, 0x20000, 0x30000, T, K, F, F, K + 24, F, L.W_KF, L.F16, 1, 0, 0, 0, C.byref(slices))
    sliced = K > (768 if T <= 2 else 1280) or F > 8192 or (K, F) == (136, 8)      # (the last: no room for the rows behind a norm)
    assert (slices.value == 1) == (not sliced)
    X, W, b = oracle.randn_f16((T, K), 1, 0, 1.0 / np.sqrt(K)), oracle.randn_f16((K, F), 2), oracle.randn_f16((F,), 3, 0, 0.02)
    R, g, beta = oracle.randn_f16((T, F), 4), oracle.randn_f16((K,), 5, 1.0, 0.1), oracle.randn_f16((K,), 6, 0, 0.1)
    held = torch.full((T, K + 24), float("nan"), dtype=torch.float16, device="cuda")
    dx = held[:, 8:8 + K]
    dx.copy_(torch.from_numpy(X))
    w, db = to_dev(W), to_dev(b)
    new = lambda dt=torch.float16: poison(torch.empty((T, F), dtype=dt, device="cuda"))
    for epi, res, dt in (("gelu", None, torch.float16), ("none", R, torch.float16), ("relu", None, torch.float32)):
        out = new(dt)
        ctx.ws.reset()
        jv.matmul_(ctx, out, w, dx, db, epi=epi, residual=None if res is None else to_dev(res))
        assert_parity(to_host(out), oracle.gemm_f16(X, W, b, epi=epi, residual=res), what=f"T{T} K{K} F{F} {epi}")
    exact = X.astype(np.float64) @ W.astype(np.float64) + b.astype(np.float64)
    out = new(torch.float32)
    ctx.ws.reset()
    jv.matmul_(ctx, out, w, dx, db)
    assert np.linalg.norm(to_host(out) - exact) <= 2.0 ** -24 * max(8.0, np.sqrt(K)) * np.linalg.norm(exact)
    h, folded, apart = torch.empty((T, K), dtype=torch.float16, device="cuda"), new(), new()
    jv.layernorm_(ctx, h, None, None, dx.contiguous(), to_dev(g), to_dev(beta), K, 1e-5)
    ctx.ws.reset()
    jv.ln_matmul_(ctx, folded, w, dx, to_dev(g), to_dev(beta), 1e-5, db)
    ctx.ws.reset()
    jv.matmul_(ctx, apart, w, h, db)
    assert torch.equal(folded, apart)


@pytest.mark.parametrize("T,K,F,dt", [(5, 8200, 17, "f16"), (8, 12296, 40, "f16"), (6, 12544, 9, "f32"), (8, 16384, 24, "f32"), (4, 16384, 24, "f16")])
def test_rows_of_the_deepest_k(ctx, T, K, F, dt):
    """mi_gemv_f16 takes [F][K] weights as deep as eight rows' share of its bound on LDS lets through, 16 384, at every T; the kernel's
    rounds end in each of the last two.  Error as in test_rows, and half a step of fp16 where the result is that.  Deeper is declined."""
    import torch
    from juliavision_amd import _lib as L
    X, W, b = oracle.randn_f16((T, K), 1, 0, 1.0 / np.sqrt(K)), oracle.randn_f16((F, K), 2), oracle.randn_f16((F,), 3, 0, 0.02)
    out = poison(torch.empty((T, F), dtype=torch.float16 if dt == "f16" else torch.float32, device="cuda"))
    dx, dw, db = to_dev(X), to_dev(W), to_dev(b)

    def gemv(k):
        return ctx.lib.mi_gemv_f16(out.data_ptr(), dx.data_ptr(), dw.data_ptr(), db.data_ptr(), None, T, k, F, F, k, k, L.W_FK, L.BIAS_COL,
                                   L.EPI["none"], L.F16 if dt == "f16" else L.F32, None, 0, ctx.stream)
    assert gemv(16384 + 8) == L.DECLINE_EXTENT            # nothing is enqueued
    assert gemv(K) == L.OK
    torch.cuda.synchronize()
    exact = X.astype(np.float64) @ W.astype(np.float64).T + b.astype(np.float64)
    err = np.linalg.norm(to_host(out).astype(np.float64) - exact) / np.linalg.norm(exact)
    assert err <= 2.0 ** -24 * np.sqrt(K) + (2.0 ** -11 if dt == "f16" else 0.0)
