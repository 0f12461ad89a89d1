"""The route of prefill-sized products on registered weights (host code, no GPU):
the tile and split the plan picks, and where the LDS tile kernel takes over."""
import ctypes
import os

import pytest

from test_gpu_prefill import GLU, PRODUCTS


@pytest.fixture(scope="module")
def plan():
    from alveare_amd import _lib, build

    if not os.path.exists(_lib.LIB_PATH):
        build.build()
    L = _lib.lib()

    def f(M, N, K, fp32=False, ffn=0):
        t, k = ctypes.c_int(), ctypes.c_int()
        assert L.alv_prefill_plan(M, N, K, int(fp32), ffn, ctypes.byref(t), ctypes.byref(k)) == 0
        return t.value, k.value

    return f


def test_cases_run_the_tiles_they_name(plan):
    """The GPU tests' products and FFNs still have the plans listed beside them,
    and together cover every tile built, unsplit and split."""
    for dtype, shapes in PRODUCTS.items():
        for M, N, K, *want in shapes:
            assert plan(M, N, K, dtype == "fp32") == tuple(want), (M, N, K, dtype)
    for M, I, H, *want in GLU:
        assert plan(M, I, H, ffn=1) == tuple(want), (M, I, H)
    tiles = {32, 64, 128, 192, 256}
    for cases in ([tuple(s[3:]) for shapes in PRODUCTS.values() for s in shapes], [s[3:] for s in GLU]):
        assert tiles <= {t for t, k in cases if k == 1}
        assert tiles <= {t for t, k in cases if k > 1}


@pytest.mark.parametrize("M,N,K,fp32,lds", [
    (17, 8192, 3840, 0, True), (64, 8192, 3840, 0, True), (65, 8192, 3840, 0, False), (333, 8192, 3840, 0, False),
    (64, 3840, 4096, 0, False), (64, 3072, 2048, 0, False), (512, 1536, 1152, 0, False), (4000, 1536, 1152, 0, True),
    (128, 256, 256, 0, True), (129, 256, 256, 0, False), (2000, 3840, 32, 0, True), (200, 3840, 32, 0, True),
    (64, 8192, 3840, 1, False), (64, 3840, 64, 1, True), (64, 3840, 96, 1, False), (2048, 3840, 256, 1, True),
    (2048, 3840, 512, 1, False)])
def test_short_products_keep_the_lds_kernel(plan, M, N, K, fp32, lds):
    """Both sides of the rule's lines at sizes where the packing launch was
    measured slower, and where it was measured faster."""
    assert (plan(M, N, K, bool(fp32)) == (0, 0)) == lds
    assert plan(M, N, K, bool(fp32), 1) != (0, 0)  # an FFN's products always pack
    assert plan(M, N, K, False, 2) != (0, 0)


def test_plan_refuses_what_no_product_has(plan):
    from alveare_amd import _lib

    L, t = _lib.lib(), ctypes.c_int()
    for M, N, K in ((0, 1, 32), (1, 0, 32), (1, 1, 0), (1, 1, 48)):
        assert L.alv_prefill_plan(M, N, K, 0, 0, ctypes.byref(t), ctypes.byref(t)) == _lib.ALV_ERR_ARG
    assert L.alv_prefill_plan(1, 1, 32, 0, 3, ctypes.byref(t), ctypes.byref(t)) == _lib.ALV_ERR_ARG
    assert L.alv_prefill_plan(1, 1, 32, 0, 0, None, ctypes.byref(t)) == _lib.ALV_ERR_ARG
