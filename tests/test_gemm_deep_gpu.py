"""The 32 x 32 kernel whose waves split K, where it can go wrong: fewer stages of K than it asks for ahead, as many as its ring and around
it, odd and even counts, a K that ends anywhere in a 128-deep stage, ragged rows and columns, its limit of one workgroup a CU,
fp32 partial planes, a folded norm's statistics wave."""
import numpy as np
import pytest

import oracle
from util import assert_parity, poison, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["kf", "fk"])
@pytest.mark.parametrize("K", [72, 128, 136, 192, 256, 384, 520, 632, 640, 768, 896, 1024, 1032, 1152, 1216, 2304])
@pytest.mark.parametrize("T,F", [(9, 64), (70, 72), (500, 504)])      # 2, 9 and 256 workgroups
def test_stages_of_k(ctx, T, F, K, layout):
    import torch
    import juliavision_amd as jv
    X, W = oracle.randn_f16((T, K), 1, 0, 1.0 / np.sqrt(K)), oracle.randn_f16((K, F), 2)
    b, R = oracle.randn_f16((F,), 3, 0, 0.02), oracle.randn_f16((T, F), 4)
    out = poison(torch.empty((T, F), dtype=torch.float16, device="cuda"))
    w = to_dev(W) if layout == "kf" else to_dev(np.ascontiguousarray(W.T)).t()
    ctx.ws.reset()
    jv.matmul_(ctx, out, w, to_dev(X), to_dev(b), residual=to_dev(R))
    torch.cuda.synchronize()
    assert_parity(to_host(out), oracle.gemm_f16(X, W, b, residual=R), what=f"T{T} K{K} F{F} {layout}")


@pytest.mark.parametrize("layout", ["kf", "fk"])
@pytest.mark.parametrize("T,K,F", [(16, 8192, 64), (256, 6016, 512), (40, 5120, 1280)])
def test_long_k(ctx, T, K, F, layout):
    """Also those whose K is split over workgroups as well."""
    import torch
    import juliavision_amd as jv
    X, W = oracle.randn_f16((T, K), 1, 0, 1.0 / np.sqrt(K)), oracle.randn_f16((K, F), 2)
    out = poison(torch.empty((T, F), dtype=torch.float16, device="cuda"))
    w = to_dev(W) if layout == "kf" else to_dev(np.ascontiguousarray(W.T)).t()
    ctx.ws.reset()
    jv.matmul_(ctx, out, w, to_dev(X))
    torch.cuda.synchronize()
    assert_parity(to_host(out), oracle.gemm_f16(X, W), what=f"T{T} K{K} F{F} {layout}")


@pytest.mark.parametrize("K", [128, 192, 320, 512, 576, 1280])
@pytest.mark.parametrize("T,F", [(33, 72), (500, 504)])
def test_folded_norm(ctx, T, F, K):
    """The statistics wave keeps the loop's barriers, whatever the count of stages."""
    import torch
    import juliavision_amd as jv
    x, W = oracle.randn_f16((T, K), 5, 1.0, 2.0), oracle.randn_f16((K, F), 6, 0, 1.0 / np.sqrt(K))
    b, g, beta = oracle.randn_f16((F,), 7, 0, 0.02), oracle.randn_f16((K,), 8, 1.0, 0.1), oracle.randn_f16((K,), 9, 0, 0.1)
    folded = jv.lnfold_prepare(ctx, to_dev(W), to_dev(g), to_dev(beta), to_dev(b))
    stats = poison(jv.rowstats_new(T, K))
    dx = to_dev(x)
    jv.rowstats_(ctx, stats, dx)
    out = poison(torch.empty((T, F), dtype=torch.float16, device="cuda"))
    jv.lnfold_matmul_(ctx, out, folded, dx, stats, 1e-5)
    torch.cuda.synchronize()
    want = oracle.gemm_f16(oracle.layernorm_f16(x, g, beta, 1e-5)[0], W, b)
    assert_parity(to_host(out), want, what=f"T{T} K{K} F{F}")
