"""Every form of the staged dense product (qw_gmm.hip k_xgemm) at the plans
that a call really gets: each tile width unsplit and split, scales that come
as one flat copy, 8 groups a load and one by one, in one window of a column's
groups, in several, and in windows cut to a slice; and a call of more rows
than are staged at a time, whose last rows have a plan of their own.  Each
case names its plan, so that a change of the rule cannot drop it unseen.

Bar as in test_gpu_qmm_tiles.py: activations carry one f16 rounding, rel-L2
about 2.1e-4 against the oracle's weights in 64 bits, 4e-4 allowed."""
import ctypes as C

import numpy as np
import pytest

from qwasar_amd import synth

pytestmark = pytest.mark.gpu

SGL = {16: 96, 32: 48, 64: 96, 128: 48}      # groups a column in LDS, by rows a tile


def plan(gpu, rows, k, n, G):
    out = (C.c_int * 4)()
    C.CDLL(gpu.LIB_PATH).qwk_qmm_plan(k, n, rows, G, out)
    return tuple(out)


def loads(k, n, G, bm):
    """How the scales come, and in how many windows a slice of all of k."""
    g = k // G
    if g <= SGL[bm] and g * n % 8 == 0:
        return "flat"
    return ("eight" if g % 8 == 0 else "one") + ("" if g <= SGL[bm] else " windows")


def rel_l2(a, b):
    a, b = np.asarray(a, np.float64).ravel(), np.asarray(b, np.float64).ravel()
    return float(np.sqrt(((a - b) ** 2).sum() / max((b * b).sum(), 1e-300)))


def product(gpu, rows, k, n, G):
    q = synth.make_q4(rows + k + n, "plan", n, k, G)
    x = np.random.default_rng(rows).uniform(-1, 1, (rows, k)).astype(np.float32)
    B = gpu.Buf
    bufs = [B.of(a) for a in (q.w, q.s, q.b, x)]
    yb = B.of(np.full((rows + 1, n), 7.0, np.float32))
    c = gpu.qw_cmd_begin()
    gpu.qw_op_qmm_q4(c, yb.ref(), bufs[3].ref(), *[b.ref() for b in bufs[:3]], k, n, rows, G)
    gpu.run(c, "qmm")
    y = yb.read(np.float32, (rows + 1, n))
    assert (y[rows] == 7.0).all(), "rows past the product are left alone"
    y = y[:rows]
    # fp32 products of the oracle's weights: 1e-6 at these k, far under the bar
    want = x @ q.dequant().astype(np.float32).T
    for r0 in range(0, rows, 128):              # a tile at a time: no tile hides behind the rest
        assert rel_l2(y[r0:r0 + 128], want[r0:r0 + 128]) < 4e-4, f"rows from {r0}"
    for c0 in range(0, n, 160):
        assert rel_l2(y[:, c0:c0 + 160], want[:, c0:c0 + 160]) < 4e-4, f"columns from {c0}"


@pytest.mark.parametrize("rows,k,n,G,tile,cols,split,how", [
    # one workgroup for all of k
    (30, 896, 5000, 64, 16, 4, False, "flat"),
    (30, 640, 7001, 128, 16, 4, False, "one"),
    (100, 896, 1500, 128, 32, 4, False, "one"),
    (100, 1568, 6150, 32, 32, 4, False, "one windows"),
    (250, 768, 700, 128, 64, 4, False, "flat"),
    (300, 640, 700, 128, 64, 4, False, "one"),
    (515, 1792, 4990, 32, 128, 2, False, "eight windows"),
    (640, 1568, 3000, 32, 128, 2, False, "one windows"),
    (900, 672, 4100, 32, 128, 3, False, "one"),
    (515, 1568, 7001, 32, 128, 3, False, "one windows"),
    (900, 640, 6150, 32, 128, 4, False, "flat"),
    (900, 1792, 6150, 32, 128, 4, False, "eight windows"),
    (1000, 3072, 10230, 64, 128, 5, False, "flat"),
    (1000, 3392, 10230, 64, 128, 5, False, "one windows"),
    (1000, 3584, 10230, 64, 128, 5, False, "eight windows"),
    # slices of whole 16-group blocks of the staged sums
    (16, 4160, 6144, 32, 16, 4, True, "one windows"),
    (16, 5632, 6144, 32, 16, 4, True, "eight windows"),
    (20, 2240, 3000, 32, 16, 4, True, "flat"),
    (100, 1344, 1000, 32, 32, 4, True, "flat"),
    (100, 1920, 700, 32, 32, 4, True, "one windows"),
    (129, 4608, 320, 32, 64, 4, True, "eight windows"),
    (129, 2336, 1090, 32, 64, 4, True, "one"),
    (700, 800, 700, 32, 128, 2, True, "one"),
    (200, 2336, 4100, 32, 128, 3, True, "one windows"),
    (900, 2816, 2050, 64, 128, 4, True, "flat"),
    (900, 3584, 2050, 64, 128, 5, True, "eight windows"),
    # and that start or end inside one
    (20, 6720, 1000, 32, 16, 4, True, "one windows"),
    (50, 1792, 1500, 128, 16, 4, True, "flat"),
    (100, 1344, 1000, 64, 32, 4, True, "flat"),
    (100, 4608, 320, 64, 32, 4, True, "eight windows"),
    (100, 1920, 700, 128, 32, 4, True, "one"),
    (200, 672, 1000, 32, 64, 4, True, "flat"),
    (129, 3264, 320, 32, 64, 4, True, "one windows"),
    (515, 1600, 320, 32, 128, 2, True, "one windows"),
    (200, 3328, 4100, 32, 128, 3, True, "eight windows"),
    (515, 4224, 2050, 128, 128, 4, True, "one"),
    (200, 4128, 6150, 32, 128, 5, True, "one windows"),
    (515, 4224, 3000, 128, 128, 5, True, "flat"),
])
def test_staged_plans(gpu, rows, k, n, G, tile, cols, split, how):
    p = plan(gpu, rows, k, n, G)
    assert (p[0], p[1], p[2] > 1, loads(k, n, G, tile)) == (tile, cols, split, how), p
    product(gpu, rows, k, n, G)


def test_more_rows_than_are_staged_at_a_time(gpu):
    """8192 rows unsplit, then 13 of their own plan, split: the partials lie
    behind the shorter stage."""
    assert plan(gpu, 8205, 2112, 520, 64)[::2] == (128, 1)
    product(gpu, 8205, 2112, 520, 64)
