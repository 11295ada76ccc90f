"""The dense 4-bit product's plan (qw_gmm.hip qx_plan) without a GPU: whole
slices that cover k, and no plan that leaves the chip idle or multiplies
mostly empty rows where a finer one is at hand."""
import ctypes as C
import math

import pytest

from qwasar_amd import gpu

SLOTS = 512          # workgroups the chip holds at two a CU


def plan(rows, k, n, G):
    out = (C.c_int * 4)()
    C.CDLL(gpu.LIB_PATH).qwk_qmm_plan(k, n, rows, G, out)
    return tuple(out)


def cut(a, b):
    return -(-a // b)


SHAPES = [(r, k, n, G) for r in (9, 17, 33, 65, 100, 129, 192, 256, 257, 400, 512, 1000, 2048)
          for k, n in ((1024, 512), (3072, 3072), (3456, 5888), (5888, 3456), (3072, 8192), (6144, 10240), (4160, 6144))
          for G in (32, 64)]


@pytest.mark.parametrize("rows,k,n,G", SHAPES)
def test_slices_are_whole_and_cover_k(rows, k, n, G):
    bm, cols, splits, ks = plan(rows, k, n, G)
    assert bm in (0, 16, 32, 64, 128) and splits >= 1 and ks >= 1
    assert cut(k, ks) == splits
    if splits > 1:
        assert ks % (8 * G if bm else 128) == 0


@pytest.mark.parametrize("rows,k,n,G", [(124, 3136, 7616, 64), (129, 3456, 5888, 64), (160, 3456, 5888, 64),
                                        (192, 3456, 5888, 64), (243, 4224, 4608, 64), (160, 4160, 6144, 32)])
def test_middle_sizes_fill_the_chip(rows, k, n, G):
    """Three workgroups for every four CUs or more: these ran on 119 to 192,
    a tenth to a fifth slower than 64 x 64 tiles in three slices."""
    bm, cols, splits, ks = plan(rows, k, n, G)
    assert bm in (32, 64, 128)
    assert cut(rows, bm) * cut(n, 32 * cols) * splits > 3 * SLOTS // 8, (bm, cols, splits, ks)


@pytest.mark.parametrize("rows,k,n,G", [s for s in SHAPES if 65 <= s[0] <= 192 and s[3] == 64])
def test_few_empty_rows(rows, k, n, G):
    """Up to 192 rows no more than 63 rows of padding (129 paid for 256)."""
    assert plan(rows, k, n, G)[0] <= 64


@pytest.mark.parametrize("k,n,pairs,E", [(640, 640, 2400, 256), (320, 640, 2400, 256), (640, 640, 360, 256),
                                         (512, 896, 1432, 256), (256, 1792, 2322, 128)])
def test_grouped_last_round_is_not_nearly_empty(k, n, pairs, E):
    """Column blocks are run back to back where k is short, but not so that a
    few workgroups are left for a round of their own (261 tiles of 5 blocks,
    three at a time: 522 workgroups, a round of 512 and one of 10)."""
    rows = gpu.qw_moe_tile_rows(pairs, E)
    w = C.CDLL(gpu.LIB_PATH).qwk_gather_gemm_blocks(k, n, pairs, E, rows)
    blocks = cut(n, 128)
    assert 1 <= w <= min(blocks, 8)
    p = [math.exp(-pairs / E)]                          # pairs an expert: Poisson
    for i in range(1, 200):
        p.append(p[-1] * pairs / E / i)
    wgs = E * sum(q * cut(i, rows) for i, q in enumerate(p)) * cut(blocks, w)
    assert wgs <= SLOTS or wgs % SLOTS >= SLOTS // 8 or wgs > 4 * SLOTS, (w, wgs)
