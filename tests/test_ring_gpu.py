"""The 64 x 64 ring kernel where it can go wrong: fewer tiles of K than it asks for ahead, as many as its ring and around it, odd and
even counts, a K that ends inside a tile, ragged rows and columns, one and two workgroups a CU, a folded norm's statistics wave."""
import numpy as np
import pytest

import oracle
from util import assert_parity, poison, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["kf", "fk"])
@pytest.mark.parametrize("K", [72, 128, 136, 192, 256, 320, 384, 448, 512, 520, 576, 640, 1096])
@pytest.mark.parametrize("T,F", [(1000, 1000), (1100, 1096)])      # 256 workgroups, and 324: more than one on a CU
def test_tiles_of_k(ctx, T, F, K, layout):
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


@pytest.mark.parametrize("K", [128, 192, 320, 512, 576, 1280])
@pytest.mark.parametrize("T,F", [(1000, 1000), (1100, 1096)])
def test_folded_norm(ctx, T, F, K):
    """The statistics wave keeps the loop's barriers, whatever the count of tiles."""
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


@pytest.mark.parametrize("T,K,F,chains", [(1000, 768, 1000, 4), (1000, 1536, 1000, 4), (300, 2304, 1000, 4), (1000, 5120, 1000, 4), (70, 3072, 768, 8), (12, 4832, 64, 16)])
def test_error_against_64_bits(ctx, T, K, F, chains):
    """fp32 results are as near as this many chains of fp32 sums leave them: 16-deep step j in chain j % chains, rounded after each half
    of it, the chains then added pairwise.  (One chain is off by 1.8 to 2 times the figure of four; a twentieth is four times the
    spread between this sum and the measured one.)  The last two are gemm_deep_kernel's."""
    import torch
    import juliavision_amd as jv
    X, W = oracle.randn_f16((T, K), 1), oracle.randn_f16((K, F), 2, 0, 1.0 / np.sqrt(K))
    out = poison(torch.empty((T, F), dtype=torch.float32, device="cuda"))
    ctx.ws.reset()
    jv.matmul_(ctx, out, to_dev(np.ascontiguousarray(W.T)).t(), to_dev(X))
    n = min(T, 96)
    x, w = X[:n].astype(np.float64), W.astype(np.float64)
    want = x @ w
    acc = np.zeros((chains, n, F), np.float32)
    for k in range(0, K, 8):
        acc[k // 16 % chains] = (acc[k // 16 % chains] + x[:, k:k + 8] @ w[k:k + 8]).astype(np.float32)
    while len(acc) > 1:
        acc = acc[::2] + acc[1::2]
    err = lambda a: np.linalg.norm(a - want) / np.linalg.norm(want)
    assert err(to_host(out)[:n].astype(np.float64)) <= 1.05 * err(acc[0].astype(np.float64))


def _kernel(T, K, F, folded=0):
    from juliavision_amd import _lib as L
    return L.GEMM_KERNELS[L.load().mi_gemm_f16_kernel(T, K, F, 1, 0, folded, None)]


RUNS = [(500, K, 520, "ring") for K in (136, 192, 256, 320, 384, 448, 512, 520, 576, 640, 1096)] + \
       [(T, K, F, "ring_shallow") for T, K, F in ((1097, 1600, 1672), (1753, 1600, 1040), (3956, 1920, 392))]


@pytest.mark.parametrize("layout", ["kf", "fk"])
@pytest.mark.parametrize("T,K,F,kernel", RUNS)
def test_the_kernel_that_is_meant(ctx, T, K, F, kernel, layout):
    """Three tiles of K (the fewest it is planned for) to eighteen, and the half ring with odd and even counts, on the kernel named."""
    import torch
    import juliavision_amd as jv
    assert _kernel(T, K, F) == kernel
    X, W = oracle.randn_f16((T, K), 1, 0, 1.0 / np.sqrt(K)), oracle.randn_f16((K, F), 2)
    b, R = oracle.randn_f16((F,), 3, 0, 0.02), oracle.randn_f16((T, F), 4)
    w = to_dev(W) if layout == "kf" else to_dev(np.ascontiguousarray(W.T)).t()
    for res, dt in ((R, torch.float16), (None, torch.float32)):
        out = poison(torch.empty((T, F), dtype=dt, device="cuda"))
        ctx.ws.reset()
        jv.matmul_(ctx, out, w, to_dev(X), to_dev(b), residual=None if res is None else to_dev(res))
        assert_parity(to_host(out), oracle.gemm_f16(X, W, b, residual=res), what=f"T{T} K{K} F{F} {layout}")


@pytest.mark.parametrize("T,K,F,kernel", [(500, K, 520, "ring") for K in (192, 320, 512, 576, 1280)] + [r for r in RUNS if r[3] == "ring_shallow"])
def test_folded_norm_on_the_kernel_that_is_meant(ctx, T, K, F, kernel):
    assert _kernel(T, K, F, 1) == kernel
    test_folded_norm(ctx, T, F, K)
