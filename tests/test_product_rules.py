"""Which kernel serves a product of many rows: the rule of csrc/gemm_tile.hip on both sides of its lines, without a GPU."""

import pytest

from clockwork_amd import ops

CUS = 256


def _choice(mode, M, N, K):
    code = ops._load("gemm_tile").cw_gemm_bf16_mid_choice(mode, M, N, K, K, CUS)
    return (code & 1023, code >> 10 & 1023, code >> 20) if code else None


# (mode, rows, N, K) where the library's product was measured to be the faster one
@pytest.mark.parametrize("mode,M,N,K", [
    # narrow outputs with a long K: a few workgroups walk the whole of it
    (0, 128, 64, 16384), (0, 144, 16, 1536), (0, 1000, 64, 1536), (0, 256, 128, 4096), (0, 144, 512, 896), (0, 700, 256, 1536),
    # tiles enough for the library
    (0, 700, 4096, 896), (0, 1500, 2048, 896), (0, 1500, 4096, 512), (0, 1000, 4096, 256), (0, 144, 2048, 1536),
    # sums for a norm: large outputs, small tiles beyond 1024 rows, whole sums of a long K, rounds that stay empty
    (3, 2048, 5120, 27648), (3, 640, 8192, 29568), (3, 2048, 8192, 29568), (3, 1434, 2048, 11008), (3, 1000, 2048, 6144), (3, 1600, 3584, 18944),
    (3, 152, 7376, 2304),
    # gated products of a narrow output
    (2, 165, 896, 4864), (2, 250, 368, 9600), (2, 92, 1280, 3072), (2, 670, 9728, 896)])
def test_products_that_stay_with_the_library(mode, M, N, K):
    assert _choice(mode, M, N, K) is None


@pytest.mark.parametrize("mode,M,N,K,wide", [
    (0, 144, 1152, 896, False), (0, 400, 2048, 1536, False), (0, 256, 64, 512, False), (0, 1000, 1152, 512, False),
    (3, 160, 1536, 8960, False), (3, 2048, 1536, 8960, True), (3, 1024, 1536, 8960, True), (3, 2048, 3584, 18944, True), (3, 256, 8192, 29568, False),
    (3, 1536, 5120, 27648, True), (3, 160, 1536, 1536, False), (3, 1000, 896, 896, False), (3, 2048, 256, 1024, False),
    (2, 160, 17920, 1536, False), (2, 400, 9728, 896, False), (2, 257, 8192, 2048, False)])
def test_products_on_the_tiles_between(mode, M, N, K, wide):
    bm, bn, planes = _choice(mode, M, N, K)
    assert (bm == 256) == wide and (planes == 1 or mode == 3)


def test_no_choice_outside_what_the_kernels_take():
    for mode in (0, 2, 3):
        for M, N, K in ((64, 1152, 896), (2049, 1152, 896), (144, 1152, 900), (144, 1152, 192), (144, 0, 896)):
            assert _choice(mode, M, N, K) is None
    assert _choice(2, 160, 9729, 896) is None and _choice(1, 160, 1152, 896) is None
