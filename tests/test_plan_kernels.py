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
