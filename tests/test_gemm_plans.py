"""The plans of the MFMA GEMM that the host makes (kernels_mfma.hip), without a device."""
import ctypes
import os
import subprocess
import sys

import pytest

import __graft_entry__ as entry

entry.load_package()
from gptrs_amd import backend  # noqa: E402

LDS = 160 * 1024   # of one CU


def lib():
    lib = backend.load_library()
    lds, part = lib._ZN5gptrs1k19mfma_int4_lds_bytesElllbm, lib._ZN5gptrs1k20mfma_workspace_bytesEilllbi   # mfma_int4_lds_bytes, mfma_workspace_bytes
    lds.argtypes, lds.restype = [ctypes.c_int64] * 3 + [ctypes.c_bool, ctypes.c_size_t], ctypes.c_size_t
    part.argtypes, part.restype = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_bool, ctypes.c_int], ctypes.c_size_t
    return lds, part


def regions(m, k, n, dual):
    """None for one launch, or (rows, columns) of the first, (row, column) of the second, the first's tile."""
    f, out = backend.load_library()._ZN5gptrs1k17mfma_bf16_regionsElllbPl, (ctypes.c_int64 * 8)()   # mfma_bf16_regions
    f.argtypes, f.restype = [ctypes.c_int64] * 3 + [ctypes.c_bool, ctypes.c_void_p], ctypes.c_int
    if f(m, k, n, dual, out) == 1:
        return None
    return (out[0], out[1]), (out[2], out[3]), (out[4], out[5])


def test_two_launches_cover_a_layer_once():
    """The first launch takes whole rows or whole columns of its tiles, the second what is left of the layer; short K stay whole."""
    two = 0
    for m in (17, 333, 600, 1000, 1713, 2047, 3000, 4758, 8188):
        for k in (64, 768, 1024, 1088, 3072, 9216):
            for n in (8, 768, 2304, 3075, 6176, 9216, 14432):
                for dual in (False, True):
                    r = regions(m, k, n, dual)
                    if r is None:
                        continue
                    (rows, cols), at, (bm, bn) = r
                    assert k > 1024 and (rows == 0) != (cols == 0) and at == (rows, cols)
                    assert rows % bm == 0 and cols % bn == 0 and rows < m and cols < n
                    two += 1
    assert two > 40


@pytest.mark.parametrize("m,k,n", [(563, 9216, 14432), (542, 11008, 14336), (352, 9216, 14432), (260, 9216, 14336), (270, 11008, 14336)])
def test_weights_that_no_cache_holds_are_not_read_again_for_a_few_rows(m, k, n):
    """Pairs of 0.5 GB of weights: one launch, or two that read half of them each."""
    r = regions(m, k, n, True)
    assert r is None or r[0][0] == 0   # (no split between rows)


@pytest.mark.parametrize("dual", [False, True])
def test_int4_tiles_fit_whatever_the_workspace(dual):
    """The scales of a workgroup's share of K lie in LDS: with the splits given up for want of room the share is all of K, and the tile has to be
    one that holds them."""
    lds, part = lib()
    split = 0
    for m in (17, 64, 200, 513, 1025, 4000):
        for k in (128, 3072, 9216, 12288, 20480, 32768, 65536, 131072, 262144):
            for n in (64, 1024, 3072, 9216):
                need = part(2, m, k, n, dual, 2)
                split += need > 0
                for room in (need, need // 2, need - 1 if need else 0, 4096, 0):
                    assert lds(m, k, n, dual, room) <= LDS, (m, k, n, room)
                assert lds(m, k, n, dual, need) == lds(m, k, n, dual, 1 << 40)      # what the planner hands in is enough for its plan
    assert split > 20


def test_the_split_switch_reaches_every_type():
    """GPTRS_HIP_GEMM_TAILSPLIT=0 (read once per process): no tile of f32, bf16 or codes is split, so none has partial sums."""
    sizes = [(d, 100, k, 768, dual, q) for d, q in ((0, 0), (2, 0), (2, 1), (2, 2)) for k in (3072, 9216) for dual in (False, True)]
    _, part = lib()
    assert all(part(*s) > 0 for s in sizes)
    code = f"import sys; sys.path[:0] = {sys.path!r}\nimport test_gemm_plans as t; part = t.lib()[1]\nprint([part(*s) for s in {sizes!r}])"
    out = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, GPTRS_HIP_GEMM_TAILSPLIT="0"), cwd=os.path.dirname(os.path.abspath(__file__)),
                         stdout=subprocess.PIPE, text=True, check=True).stdout
    assert out.strip() == str([0] * len(sizes))


# us, measured in this many splits and in those that a plan gave which took a pair for two workgroups to a CU and a second workgroup on a CU for nothing
@pytest.mark.parametrize("m,k,n,dual,splits", [(333, 768, 768, False, 3),     # 11.5, in 6 13.0
                                               (640, 768, 768, False, 2),     # 14.0, in 4 15.5
                                               (200, 1024, 1024, False, 4),   # 12.7, in 8 14.1
                                               (200, 768, 3072, True, 1),     # 26.1, in 2 32.9
                                               (200, 1024, 2816, True, 1)])   # 31.9, in 2 38.7
def test_f32_as_bf16_products_is_split_where_it_pays(m, k, n, dual, splits):
    assert lib()[1](0, m, k, n, dual, 0) == (splits > 1) * splits * m * n * 4 * (1 + dual)


class SkinnyPlan(ctypes.Structure):
    _fields_ = [("nw", ctypes.c_int), ("depth", ctypes.c_int), ("ks", ctypes.c_int)]


# waves, requests of a wave and splits of layers of 2 to 16 rows where they were measured (us, and with the choice made before)
@pytest.mark.parametrize("f32,m,k,n,dual,want", [(0, 12, 4096, 11008, True, (8, 1, 1)),    # 29.6, 16 waves of one 36.9
                                                 (0, 12, 768, 50257, True, (8, 2, 1)),     # 26.2, 16 of one 32.2
                                                 (0, 8, 512, 32000, False, (8, 2, 1)),     # 8.5, 8 of four 11.0
                                                 (0, 12, 4096, 1024, True, (8, 2, 2)),     # 8.2, 16 of one, unsplit 11.9
                                                 (1, 12, 2048, 8192, False, (8, 1, 1)),    # 14.9, 16 of one 16.9
                                                 (1, 8, 3072, 576, True, (16, 2, 4)),      # 8.7, in two 10.7
                                                 (1, 12, 4096, 11008, True, (16, 1, 1)),   # 62.3, 8 of one 67.3
                                                 (0, 12, 3072, 32768, False, (16, 1, 1)),  # 37.1, 8 of two 40.4
                                                 (0, 8, 9216, 3072, False, (16, 2, 1)), (1, 8, 3072, 768, False, (16, 2, 2)), (1, 7, 768, 50257, False, (8, 4, 1))])
def test_layers_of_few_rows(f32, m, k, n, dual, want):
    plan = backend.load_library()._ZN5gptrs1k11skinny_planEilllbb
    plan.argtypes, plan.restype = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_bool] * 2, SkinnyPlan
    p = plan(0 if f32 else 2, m, k // (16 if f32 else 32), n, dual, False)
    assert (p.nw, p.depth, p.ks) == want
