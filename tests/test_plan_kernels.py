"""Which kernel runs, asked on the CPU: the answer follows the path (the precision) that the plan names, over the forms a call can take."""
import ctypes as C
import itertools

import pytest

from juliavision_amd import _lib as L

PTR = 0x10000
OF_PATH = {"decline": {"none"}, "flash": {"fused", "tiles"}, "rows": {"tiles_f32", "rows", "one_query"}}


def _sdpa(E, Lq, Lk, H, B, *, packed=False, mask=None, q=PTR, out=None, out_strides=None, f32=False):
    row = 3 * H * E if packed else E
    st = (lambda n: L.strides4(1, row, E, row * n)) if packed else (lambda n: L.strides4(1, E, E * n, E * n * H))
    ns, nsplit = C.c_int(0), C.c_int(0)
    path = L.load().mi_sdpa_f16_plan(q, st(Lq), PTR, st(Lk), PTR, st(Lk), int(mask is not None), 0, E, Lq, Lk, H, B, 0.125, C.byref(ns))
    bst = {None: None, "key": L.strides4(1, 0, 0, Lk), "dense": L.strides4(1, Lk, Lk * Lq, Lk * Lq * H), "key32": L.strides4(1, 0, 0, Lk)}[mask]
    kernel = L.load().mi_sdpa_f16_kernel(out, L.F32 if f32 else L.F16, out_strides, q, st(Lq), PTR, st(Lk), PTR, st(Lk), None if mask is None else PTR,
                                         L.F32 if mask == "key32" else L.F16, bst, E, Lq, Lk, H, B, 0.125, C.byref(nsplit))
    return L.SDPA_PATHS[path], L.SDPA_KERNELS[kernel], ns.value, nsplit.value


@pytest.mark.parametrize("packed", [False, True])
def test_the_kernel_is_one_of_the_plans_path(packed):
    seen = set()
    for E, Lq, Lk, (H, B), mask in itertools.product([16, 20, 32, 40, 64, 72, 80, 128, 160, 256], [1, 2, 7, 23, 63, 64, 128, 700, 4096],
                                                     [1, 16, 64, 300, 1500, 4096, 8192], [(1, 1), (8, 1), (20, 4)], [None, "key", "dense"]):
        path, kernel, plan_splits, splits = _sdpa(E, Lq, Lk, H, B, packed=packed, mask=mask)
        if mask == "key" and path == "rows" and Lq >= 64:                      # the plan sees a dense mask, whose rows may start off 4 bytes
            assert kernel in OF_PATH["flash"] | OF_PATH["rows"]
        else:
            assert kernel in OF_PATH[path], (E, Lq, Lk, H, B, mask)
        assert splits <= max(plan_splits, 1), (E, Lq, Lk, H, B, mask)             # the workspace has room for the plan's
        seen.add(kernel)
    assert seen == {"none"} | OF_PATH["flash"] | OF_PATH["rows"] or seen == OF_PATH["flash"] | OF_PATH["rows"]


def test_which_kernel_a_gemm_runs():
    kernel = lambda T, K, F, epi="none", folded=0: L.GEMM_KERNELS[L.load().mi_gemm_f16_kernel(T, K, F, 1, L.EPI[epi], folded, None)]
    for K in (72, 128, 256, 512, 520, 1024, 2304):           # few tiles: 32 x 32 ones, K in one chain up to 512
        assert kernel(9, K, 64) == kernel(70, K, 72) == ("deep" if K > 512 else "deep_serial")
    for K in (520, 640, 768, 1152, 2304):
        assert kernel(500, K, 504) == "deep" and kernel(500, K, 520) == "ring"      # 256 tiles of 32 x 32, and more
    assert kernel(1500, 1280, 5120, "gelu") == "wide" and kernel(1544, 1288, 1288) == "staged" and kernel(1500, 5120, 1280) == "exchange"
    assert kernel(2012, 1280, 1152) == kernel(2012, 1280, 1152, "relu") == "staged" and kernel(4510, 2048, 1280) == "wide"
    # past the four-wave tiles' first choice: narrow ones at K of two and three tiles, square ones at a long K
    assert kernel(6637, 128, 1360) == kernel(7310, 192, 1304) == kernel(3399, 256, 2312) == kernel(3376, 2560, 624) == "staged"
    assert kernel(1808, 128, 3952) == kernel(2447, 128, 2816) == kernel(4525, 192, 1688) == kernel(1571, 1024, 2544) == "wide"
    assert kernel(8, 1280, 1280) == kernel(100, 1284, 64) == "none" and kernel(100, 64, 64) == "one_tile"
    # a GELU moves a call only between tiles that sum K in one order
    for T, K, F in itertools.product((70, 300, 500, 1000, 1370, 3000), (384, 520, 1024, 1536, 2304), (64, 384, 520, 1536, 4096)):
        plain, gelu = kernel(T, K, F), kernel(T, K, F, "gelu")
        own = {"ring", "ring_shallow", "deep", "exchange"}
        if K > 512:
            assert (plain in own) == (gelu in own) and (plain not in own or plain == gelu), (T, K, F)


@pytest.mark.parametrize("T,K,F,runs", [(1181, 896, 3264, "wide"), (4665, 896, 784, "wide"), (4665, 640, 784, "staged"), (2518, 192, 3552, "staged")])
def test_narrow_tiles_end_at_k_768(T, K, F, runs):
    """Two workgroups a CU of 64 x 128 tiles, whose estimate is lowered up to there."""
    assert L.GEMM_KERNELS[L.load().mi_gemm_f16_kernel(T, K, F, 1, L.EPI["none"], 0, None)] == runs


def test_how_rows_against_kf_weights_are_cut():
    """One slice of K where they run as 32 x 32 tiles, which ask for row pitches below 2^31 bytes a tile."""
    slices = C.c_int(0)

    def cut(T, K, F, ldX=None, ldW=None):
        assert L.GEMM_PATHS[L.load().mi_gemm_f16_plan_caps(None, PTR, PTR, PTR, T, K, F, F, ldX or K, ldW or F, L.W_KF, L.F16, 1, 0, 0, 0, C.byref(slices))] == "skinny"
        return slices.value
    assert cut(1, 384, 1536) == cut(8, 1280, 5120) == cut(2, 768, 768) == 1
    assert cut(1, 776, 768) > 1 and cut(8, 1288, 5120) > 1 and cut(4, 128, 8200) > 1
    assert cut(1, 384, 1536, ldX=2 ** 25 - 8, ldW=2 ** 23 - 8) == 1 and cut(1, 384, 1536, ldX=2 ** 25) > 1 and cut(1, 384, 1536, ldW=2 ** 23) > 1


def test_which_kernel_gathers_patches():
    def kernel(H, W, Cin, Cout, k, s=1, groups=1):
        args = (W, H, Cin, 1, k, k, Cout, s, s, k // 2, k // 2, 1, 1, groups)
        conv, gemm = L.CONV_KERNELS[L.load().mi_conv2d_f16_kernel(*args, None)], L.GEMM_KERNELS[L.load().mi_conv2d_f16_patch_kernel(*args)]
        assert (gemm == "none") == (conv != "patch_gemm")
        return gemm
    assert kernel(22, 23, 96, 96, 5) == "deep" and kernel(64, 64, 256, 256, 3) == "ring" and kernel(128, 128, 256, 256, 3) == "ring_shallow"
    assert kernel(64, 64, 256, 256, 1) == kernel(64, 64, 256, 256, 3, groups=4) == kernel(1024, 1024, 3, 144, 7, 4) == "none"


def test_what_the_tiles_do_not_take():
    assert _sdpa(64, 256, 256, 8, 4)[1] == "tiles"
    assert _sdpa(64, 256, 256, 8, 4, q=PTR + 2)[1] == "rows"                       # off 16 bytes
    assert _sdpa(64, 256, 256, 8, 4, out=PTR + 2)[1] == "rows"
    assert _sdpa(64, 256, 256, 8, 4, mask="dense")[1] == "fused" and _sdpa(64, 256, 256, 8, 4, mask="key32")[1] == "fused"
    assert _sdpa(64, 256, 5000, 8, 4, mask="key")[1] in ("fused", "rows")          # a mask row longer than its LDS
    assert _sdpa(80, 256, 256, 8, 4)[1] == "fused"                                 # a head size without chunk permutations
    assert _sdpa(64, 23, 300, 8, 2)[1] == _sdpa(64, 23, 300, 8, 2, f32=True)[1] == "tiles_f32"
    assert _sdpa(72, 23, 300, 8, 2)[1] == "tiles_f32" and _sdpa(72, 23, 300, 8, 2, f32=True)[1] == "rows"
    assert _sdpa(64, 23, 300, 8, 2, mask="key")[1] == "tiles_f32" and _sdpa(64, 23, 300, 8, 2, mask="key32")[1] == "rows"
    assert _sdpa(64, 1, 1500, 20, 1)[1:] == ("one_query", 4, 4)
    # 2^25 workgroups of 128 threads are more than one launch dimension holds
    assert _sdpa(16, 2, 64, 512, 65535)[1] == "tiles_f32" and _sdpa(16, 2, 64, 520, 65535)[1] == "rows"
    assert _sdpa(16, 128, 64, 128, 65535)[1] == "tiles" and _sdpa(16, 128, 64, 130, 65535)[1] == "fused"


def test_the_largest_image_of_the_patch_gather():
    """Its byte offsets are 32 bits and are raised by up to 3072 on their way into the loads."""
    kernel = lambda h: L.CONV_KERNELS[L.load().mi_conv2d_f16_kernel(47, h, 256, 1, 3, 3, 512, 4, 4, 0, 0, 1, 1, 1, C.byref(C.c_size_t(0)))]
    assert 47 * 178481 * 256 > 2 ** 31 - 1536 > 47 * 178480 * 256
    assert kernel(178480) == "patch_gemm" and kernel(178481) == "im2col_gemm"


def test_maps_whose_matrix_cannot_be_staged_run_in_one_launch():
    """Patches that do not overlap, their im2col matrix beyond 32-bit extents: the staged route would refuse them."""
    for H, Cout, k in ((26000, 64, 14), (26000, 12, 2), (26700, 64, 15)):
        scratch = C.c_size_t(1)
        assert L.CONV_KERNELS[L.load().mi_conv2d_f16_kernel(H, H, 3, 1, k, k, Cout, k, k, 0, 0, 1, 1, 1, C.byref(scratch))] == "tile" and scratch.value == 0


def test_the_workspace_covers_whichever_convolution_kernel_runs():
    import random
    rng, lib, seen = random.Random(0), L.load(), set()
    for i in range(4000):
        k, groups = rng.choice([1, 3, 3, 5, 7, 26]), rng.choice([1, 1, 1, 4])
        cin, cout = (rng.choice([1, 3, 16, 32, 64, 70, 96, 128, 256]) * groups, rng.choice([1, 6, 32, 64, 96, 256]) * groups)
        w, h, s, p = rng.randint(1, 200), rng.randint(1, 200), rng.choice([1, 1, 2, 4]), rng.choice([0, k // 2])
        args = (w, h, cin, rng.choice([1, 2]), k, k, cout, s, s, p, p, 1, 1)
        need = C.c_size_t(0)
        kernel = L.CONV_KERNELS[lib.mi_conv2d_f16_kernel(*args, groups, C.byref(need))]
        path = L.CONV_PATHS[lib.mi_conv2d_f16_plan(*args, groups)]
        assert (kernel == "none") == (path == "decline") and (kernel == "direct") == (path == "direct") and (kernel == "gemm_1x1") == (path == "gemm_1x1")
        assert need.value <= lib.mi_conv2d_f16_workspace(*args), args
        seen.add(kernel)
    assert seen == set(L.CONV_KERNELS.values())
