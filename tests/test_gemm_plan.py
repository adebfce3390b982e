"""The GEMMs' plans (which kernel, tiles and shares of K a shape takes), without a GPU."""
import ctypes

import pytest

from conftest import load_host

FIELDS = ["ksplit", "wpg", "cpb", "kw", "xd", "bands", "stream", "few"]


class Plan(ctypes.Structure):
    """GemmPlan (dspark_internal.h)."""
    _fields_ = [(f, ctypes.c_int) for f in FIELDS]


def plan(M, N, K, i8=True, split=False, wpg=0, xop=False, bands=1, gs=False, rows=True, x8=False):
    """rows: x and w row-major on 16-byte boundaries."""
    p = Plan(1, 1, 4, 0, 0, 1, 0, 0)
    host = load_host()
    f = getattr(host.lib(), "_ZN6dspark9gemm_planEiiibbPNS_8GemmPlanEibibbb")
    f.argtypes = [ctypes.c_int] * 3 + [ctypes.c_bool] * 2 + [ctypes.POINTER(Plan), ctypes.c_int, ctypes.c_bool, ctypes.c_int] + \
        [ctypes.c_bool] * 3
    f.restype = None
    f(M, N, K, i8, split, ctypes.byref(p), wpg, xop, bands, gs, rows, x8)
    return p


@pytest.mark.parametrize("x8", [False, True])
@pytest.mark.parametrize("rows,xop,wpg,bands", [(True, False, 0, 1), (False, False, 0, 1), (False, True, 0, 1),
                                                (False, True, 0, 2), (False, True, 3, 1)])
def test_group_scale_ranges(rows, xop, wpg, bands, x8):
    """Ranges of K under group scales hold whole groups (two 64-column chunks), and none is empty: an idle range's waves
    would take part in every barrier and in the sum."""
    for N in (48, 512, 2048, 3072, 4096, 6144, 8208, 9984, 16464, 65520):
        for K in range(128, 8193, 128):
            for M in (1, 4, 9, 16):
                p = plan(M, N, K, wpg=wpg, xop=xop, bands=bands, gs=True, rows=rows, x8=x8)
                if p.kw == 0 or p.few:
                    continue
                band = (K // 64 + p.bands - 1) // p.bands
                per = (band + p.kw - 1) // p.kw
                per += per & 1
                assert (p.bands == 1 or band % 2 == 0) and (p.kw - 1) * per < band, (M, N, K, p.kw, per, band)


@pytest.mark.parametrize("M", [1, 8, 16])
def test_streamed_group_scales(M):
    """Row-major group scales over more tiles (64 rows) than workgroups: streamed where a tile is whole turns of the 8-slot
    ring (128 columns a step), or K is past what the K-sliced kernel holds in LDS."""
    for N in (16400, 20480, 65536, 128000):
        for K in range(128, 4609, 128):
            assert bool(plan(M, N, K, gs=True).stream) == (K % 1024 == 0 or K > 2048), (N, K)
    for K in (256, 640, 2048, 2304):
        assert plan(M, 16384, K, gs=True).stream == 4


def test_few_rows():
    """Row-major group scales up to 4096 rows: groups of 8 rows, two to a workgroup past 2048 rows; fp16 x then only up to K
    1024 or 3 tokens."""
    for M in range(1, 17):
        for N in (16, 512, 2048, 2064, 3072, 4096, 4112):
            for K in range(128, 8193, 128):
                two = N > 2048
                for x8 in (False, True):
                    want = N <= 4096 and (x8 or not two or K <= 1024 or M <= 3)
                    p = plan(M, N, K, gs=True, x8=x8)
                    assert bool(p.few) == want, (M, N, K, x8)
                    assert not want or p.wpg == 1 + two and p.kw == min(16 // p.wpg, K // 128)


def test_streamed_row_scales():
    """Row-major row scales without a split of K: the fewest tiles (4 or 8 strips) that are streamed."""
    for M, K, tiles in ((1, 2048, 192), (10, 512, 192), (11, 1792, 128), (11, 2048, 129), (15, 2048, 129), (16, 1024, 128), (16, 2048, 128),
                        (17, 1024, 128), (17, 1152, 129), (32, 2048, 129), (32, 2176, 128), (33, 2048, 96), (48, 4096, 96)):
        assert not plan(M, 64 * tiles - 64, K, split=True).stream, (M, K)
        assert plan(M, 64 * tiles, K, split=True).stream == 4 and plan(M, 64 * tiles, K, split=True).ksplit == 1, (M, K)
    for K in (128, 512, 2048, 4096):
        assert plan(49, 16, K, split=True).stream == 4 and plan(64, 4096, K, split=True).stream == 4
    for K in (64, 192):  # no whole 128-byte steps
        assert not plan(16, 65536, K, split=True).stream
