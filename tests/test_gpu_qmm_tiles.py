"""The staged 4-bit products (qw_gmm.hip) at the edges of their plans: row and
column remainders of every tile height, k that is no whole number of stages
(of 64, 128 or 256) or of 16-group blocks, split k, scale rows that come as
one flat copy, 8 groups a load or one by one (group counts past what LDS
holds, banks off a 16-byte boundary, odd group counts), and inputs whose
magnitude or layout the staging has to survive.  (Each form of the plan by
name, unsplit and reloaded ones too: test_gpu_qmm_plans.py.)

Bar: the weights enter exactly and the activations carry one f16 rounding
(relative 2^-11 at most, 2^-13 rms), so rel-L2 against the fp32 oracle is
about 2.1e-4; 4e-4 is bounded by twice that."""
import ctypes as C

import numpy as np
import pytest

from oracle import ref
from qwasar_amd import synth

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    a, b = np.asarray(a, np.float64).ravel(), np.asarray(b, np.float64).ravel()
    return float(np.sqrt(((a - b) ** 2).sum() / max((b * b).sum(), 1e-300)))


def want(q, x, rows=slice(None)):
    return np.asarray(x[rows], np.float64) @ q.dequant().astype(np.float64).T


def put(gpu, a, off):
    """A buffer holding `a` at byte `off`."""
    b = gpu.Buf(off + a.nbytes)
    b.write(a, off)
    return b


@pytest.mark.parametrize("rows,k,n,G,off", [
    (129, 1088, 1090, 64, 0),     # one row past a tile, 17 groups (odd: one by one), ragged columns
    (65, 3136, 1000, 64, 0),      # 49 groups in slices of 8: one by one, the last slice one group
    (300, 3328, 640, 64, 0),      # 52 groups, a multiple of 4, in slices of 8
    (257, 4096, 512, 64, 0),      # 64 groups in eight slices, flat; one row past a tile
    (200, 4096, 900, 128, 0),     # groups of 128
    (140, 2080, 1030, 32, 0),     # groups of 32, 65 of them, k % 64 = 32, one by one
    (16, 6144, 3000, 64, 0),      # one 16-row tile, flat scales
    (9, 8192, 4096, 32, 0),       # 256 groups of 32, 8 a load, slices of 32
    (17, 6144, 3072, 64, 0),      # 32-row tile, 8 a load
    (40, 6176, 1500, 32, 0),      # two 32-row tiles, k % 128 = 32
    (130, 3072, 700, 64, 2),      # scales and biases 2 bytes off: one by one
    (48, 3072, 2000, 64, 8),      # and 8 bytes off
    (300, 12288, 320, 64, 0),     # split k
])
def test_staged_product_edges(gpu, rows, k, n, G, off):
    q = synth.make_q4(rows + k, "edge", n, k, G)
    x = np.random.default_rng(rows).uniform(-1, 1, (rows, k)).astype(np.float32)
    B = gpu.Buf
    wb, sb, bb, xb = B.of(q.w), put(gpu, q.s, off), put(gpu, q.b, off), B.of(x)
    yb = B.of(np.full((rows + 1, n), 7.0, np.float32))
    c = gpu.qw_cmd_begin()
    gpu.qw_op_qmm_q4(c, yb.ref(), xb.ref(), wb.ref(), sb.ref(off), bb.ref(off), k, n, rows, G)
    gpu.run(c, "qmm")
    y = yb.read(np.float32, (rows + 1, n))
    assert (y[rows] == 7.0).all(), "rows past the product are left alone"
    assert rel_l2(y[:rows], want(q, x)) < 4e-4


def test_staged_product_magnitudes(gpu):
    """Each row carries its own power of two: rows of 1e6 and 1e-6, a zero
    row, a row with one large element; biases that are not -8 scales."""
    rows, k, n, G = 160, 2048, 768, 64
    q = synth.make_q4(5, "mag", n, k, G)
    q.b[:] = synth.to_bf16(np.random.default_rng(1).uniform(-3, 3, q.b.shape).astype(np.float32))
    x = np.random.default_rng(2).standard_normal((rows, k)).astype(np.float32)
    x[1] *= 1e6
    x[2] *= 1e-6
    x[3] = 0.0
    x[4, 77] = 3000.0
    B = gpu.Buf
    wb, sb, bb, xb, yb = B.of(q.w), B.of(q.s), B.of(q.b), B.of(x), B(rows * n * 4)
    c = gpu.qw_cmd_begin()
    gpu.qw_op_qmm_q4(c, yb.ref(), xb.ref(), wb.ref(), sb.ref(), bb.ref(), k, n, rows, G)
    gpu.run(c, "qmm")
    y, w = yb.read(np.float32, (rows, n)), want(q, x)
    assert (y[3] == 0.0).all()
    for r in (0, 1, 2, 4, 159):
        assert rel_l2(y[r], w[r]) < 6e-4, f"row {r}"      # one row: the rms bound above scatters by 1/sqrt(n)
    # a row of non-finite inputs stays its own
    x[9, 3] = np.nan
    x[10, 4] = np.inf
    xb.write(x)
    c = gpu.qw_cmd_begin()
    gpu.qw_op_qmm_q4(c, yb.ref(), xb.ref(), wb.ref(), sb.ref(), bb.ref(), k, n, rows, G)
    gpu.run(c, "qmm")
    y2 = yb.read(np.float32, (rows, n))
    assert not np.isfinite(y2[9]).any() and not np.isfinite(y2[10]).any()
    keep = [r for r in range(rows) if r not in (9, 10)]
    assert np.array_equal(y2[keep].view(np.uint32), y[keep].view(np.uint32))


@pytest.mark.parametrize("E,K,rows,k,n,G,by_pair", [
    (64, 4, 33, 672, 200, 32, False),     # 16-row tiles, 21 groups (odd), k % 256 != 0, ragged columns
    (64, 4, 33, 640, 2560, 32, True),     # several column blocks a workgroup
    (16, 4, 61, 2560, 100, 32, False),    # 32-row tiles, 80 groups: more than their LDS holds
    (8, 2, 130, 1152, 260, 128, True),    # 64-row tiles, groups of 128
    (32, 8, 5, 3136, 130, 64, False),     # 49 groups, 16-row tiles
])
def test_grouped_product_edges(gpu, E, K, rows, k, n, G, by_pair):
    pairs = rows * K
    q = synth.make_q4(E + k, "gedge", E * n, k, G)
    g = np.random.default_rng(pairs)
    x = g.uniform(-1, 1, (pairs if by_pair else rows, k)).astype(np.float32)
    idx = np.stack([g.choice(E, K, replace=False) for _ in range(rows)]).astype(np.int32)
    B = gpu.Buf
    wb, sb, bb, xb, ib = B.of(q.w), B.of(q.s), B.of(q.b), B.of(x), B.of(idx)
    perm, cur, tiles = B(pairs * 4), B(E * 4), B((1 + 3 * gpu.qw_moe_max_tiles(pairs, E)) * 4)
    yb = B(pairs * n * 4)
    c = gpu.qw_cmd_begin()
    gpu.qw_op_moe_group(c, perm.ref(), tiles.ref(), cur.ref(), ib.ref(), pairs, E)
    gpu.qw_op_qmm_q4_gather(c, yb.ref(), xb.ref(), perm.ref(), tiles.ref(), wb.ref(), sb.ref(), bb.ref(), k, n, pairs,
                            E, K, by_pair, G)
    gpu.run(c, "gather")
    y = yb.read(np.float32, (pairs, n))
    flat = idx.ravel()
    for e in range(E):
        p = np.flatnonzero(flat == e)
        if p.size:
            w = x[p if by_pair else p // K].astype(np.float64) @ q.dequant(e * n, n).astype(np.float64).T
            assert rel_l2(y[p], w) < 4e-4, f"expert {e}"


@pytest.mark.parametrize("rows,k,n,G", [
    (16, 4160, 6144, 32),      # 130 groups in slices of 16: a window no wider than the slice
    (24, 5632, 1536, 32),      # 176: the same, 8 a load
    (40, 4160, 6140, 32),
    (1000, 3392, 10230, 64),   # 53 groups, unsplit: two windows of 48
])
def test_staged_product_scale_windows(gpu, rows, k, n, G):
    """Scales that come by the window, few or one at a time."""
    q = synth.make_q4(rows + k, "window", n, k, G)
    x = np.random.default_rng(rows).uniform(-1, 1, (rows, k)).astype(np.float32)
    B = gpu.Buf
    wb, sb, bb, xb, yb = B.of(q.w), B.of(q.s), B.of(q.b), B.of(x), B(rows * n * 4)
    c = gpu.qw_cmd_begin()
    gpu.qw_op_qmm_q4(c, yb.ref(), xb.ref(), wb.ref(), sb.ref(), bb.ref(), k, n, rows, G)
    gpu.run(c, "qmm")
    y, w = yb.read(np.float32, (rows, n)), want(q, x)
    for c0 in range(0, n, 128):
        assert rel_l2(y[:, c0:c0 + 128], w[:, c0:c0 + 128]) < 4e-4, f"columns from {c0}"


@pytest.mark.parametrize("E,K,rows,k,n,G,by_pair", [
    (64, 4, 33, 288, 200, 32, False),     # 9 groups, k % 128 = 32, ragged columns
    (256, 6, 100, 320, 640, 64, True),
    (37, 2, 9, 256, 70, 128, True),       # tiles of one pair
    (16, 4, 40, 64, 64, 64, False),       # one stage of half a block; 10 pairs an expert
])
def test_grouped_short_k(gpu, E, K, rows, k, n, G, by_pair):
    """The unstaged form: rows as f16 holds them, and tiles with a row outside
    2^-8 .. 65504 done over with that row scaled: rows of 1e6, 1e-6, 1e-30, just
    either side of both limits, zeros, and one not finite that stays its own.
    Bar: one row's rounding error is under 6e-4 (above); f16's step of 2^-24 in
    a row whose largest is 2^-8 adds under 2^-25 / 2^-9.2, its rms, 2e-5."""
    pairs = rows * K
    assert C.CDLL(gpu.LIB_PATH).qwk_gather_gemm_small(k, n, pairs, E, gpu.qw_moe_tile_rows(pairs, E))
    q = synth.make_q4(E + k, "gshort", E * n, k, G)
    g = np.random.default_rng(pairs)
    src = pairs if by_pair else rows
    x = g.uniform(-1, 1, (src, k)).astype(np.float32)
    x[:, 0] = 1.0
    for r, m in enumerate((1e6, 1e-6, 1e-30, 65504.0, 65520.0, 2.0 ** -8, 2.0 ** -8.01, 0.0)):
        x[r] *= np.float32(m)
    idx = np.stack([g.choice(E, K, replace=False) for _ in range(rows)]).astype(np.int32)
    B = gpu.Buf
    wb, sb, bb, ib = B.of(q.w), B.of(q.s), B.of(q.b), B.of(idx)
    perm, cur, tiles = B(pairs * 4), B(E * 4), B((1 + 3 * gpu.qw_moe_max_tiles(pairs, E)) * 4)

    def product(x):
        xb, yb = B.of(x), B(pairs * n * 4)
        c = gpu.qw_cmd_begin()
        gpu.qw_op_moe_group(c, perm.ref(), tiles.ref(), cur.ref(), ib.ref(), pairs, E)
        gpu.qw_op_qmm_q4_gather(c, yb.ref(), xb.ref(), perm.ref(), tiles.ref(), wb.ref(), sb.ref(), bb.ref(), k, n,
                                pairs, E, K, by_pair, G)
        gpu.run(c, "gather")
        return yb.read(np.float32, (pairs, n))

    y = product(x)
    flat, of = idx.ravel(), np.arange(pairs) if by_pair else np.arange(pairs) // K
    for p in range(pairs):
        if p < 12 * K or p % 7 == 0:
            w = q.dequant(flat[p] * n, n).astype(np.float64) @ x[of[p]].astype(np.float64)
            assert rel_l2(y[p], w) < 7e-4, (p, of[p])
    x[8, 3] = np.inf
    y2 = product(x)
    assert not np.isfinite(y2[of == 8]).any()
    assert np.isfinite(y2[of != 8]).all()
    # a row's bits are its own, whatever else is in its tile
    x[:8] = x[9:17] if src > 17 else 1.0
    y3 = product(x)
    assert np.array_equal(y2[of > 8].view(np.uint32), y[of > 8].view(np.uint32))
    assert np.array_equal(y3[of > 8].view(np.uint32), y[of > 8].view(np.uint32))
