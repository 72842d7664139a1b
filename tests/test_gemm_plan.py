"""Which GEMM tile the bf16 projections take and in how many column ranges
(jm_gemm_plan), on the host: at the sizes whose times stand beside the rule,
the kernel that measured faster there, or within 2% of it; and the products
that are no GEMMs."""

import ctypes

import pytest

from joule_amd import _lib

NARROW, WIDE = 0, 1

QWEN3_QKV, QWEN3_O = ((4096, 512, 512), 2048), ((2048, 0, 0), 4096)
DENSE_QKV, DENSE_O = ((4096, 1024, 1024), 4096), ((4096, 0, 0), 4096)
DENSE_GU, DENSE_DN = ((12288, 12288, 0), 4096), ((4096, 0, 0), 12288)
OLMOE_QKV, OLMOE_O = ((2048, 2048, 2048), 2048), ((2048, 0, 0), 2048)


def plan(rows, K, B):
    kz = ctypes.c_int(-1)
    return _lib.lib().jm_gemm_plan(*rows, K, B, ctypes.byref(kz)), kz.value


@pytest.fixture(autouse=True)
def _built():
    if not _lib.LIB_PATH.exists():
        pytest.skip("libjoule_amd.so not built")


@pytest.mark.parametrize("shape,B,want", [
    (QWEN3_QKV, 33, (NARROW, 4)), (QWEN3_QKV, 128, (NARROW, 2)), (QWEN3_QKV, 384, (NARROW, 1)), (QWEN3_QKV, 512, (WIDE, 2)),
    (QWEN3_O, 256, (NARROW, 4)), (QWEN3_O, 512, (NARROW, 2)),
    (DENSE_QKV, 128, (NARROW, 2)), (DENSE_QKV, 129, (WIDE, 4)), (DENSE_QKV, 301, (NARROW, 1)), (DENSE_QKV, 512, (WIDE, 2)),
    (DENSE_O, 256, (NARROW, 2)), (DENSE_O, 301, (WIDE, 4)), (DENSE_O, 512, (NARROW, 1)),
    (DENSE_GU, 33, (WIDE, 4)), (DENSE_GU, 64, (NARROW, 1)), (DENSE_GU, 65, (WIDE, 2)), (DENSE_GU, 129, (WIDE, 4)),
    (DENSE_GU, 257, (WIDE, 1)), (DENSE_GU, 512, (WIDE, 2)),
    (DENSE_DN, 256, (NARROW, 2)), (DENSE_DN, 257, (WIDE, 4)), (DENSE_DN, 512, (WIDE, 4)),
    (OLMOE_QKV, 320, (NARROW, 1)), (OLMOE_QKV, 448, (WIDE, 2)), (OLMOE_O, 512, (NARROW, 2)),
])
def test_plan_follows_the_measured_times(shape, B, want):
    assert plan(*shape, B) == want


def test_plan_keeps_whole_tiles():
    """128-row matrices never take the 256-row tile, and every plan's ranges
    are whole pairs of 64-column stages."""
    for rows in ((128, 0, 0), (4096, 128, 128), (12288 + 128, 12288 + 128, 0)):
        assert all(plan(rows, 4096, B)[0] == NARROW for B in (33, 64, 200, 512, 4000))
    for K in (128, 256, 384, 512, 1024, 8192):
        for B in (33, 100, 257, 512, 5000):
            for rows in ((256, 0, 0), (24576, 256, 512)):
                kernel, kz = plan(rows, K, B)
                assert kernel in (NARROW, WIDE) and kz in (1, 2, 4) and K % (128 * kz) == 0


@pytest.mark.parametrize("rows,K,B", [((4096, 0, 0), 4096, 32), ((4096, 0, 0), 4096, 0), ((4096, 0, 0), 192, 64),
                                      ((192, 0, 0), 4096, 64), ((0, 0, 0), 4096, 64), ((128, -128, 0), 4096, 64),
                                      ((128, 0, 0), -128, 64), ((2 ** 31 - 128, 128, 0), 128, 64)])
def test_no_gemm(rows, K, B):
    kernel, kz = plan(rows, K, B)
    assert kernel == -2 and kz == -1
    assert _lib.lib().jm_gemm_plan(*rows, K, B, None) == -2
