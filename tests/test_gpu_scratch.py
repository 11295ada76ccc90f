"""Products and delta rules whose scratch cannot be had: the kernels' entry
points without their work memory, against the same calls with it through the
C ABI.  They run slower then, and are not refused.

Bars: either form of a product is within 4e-4 of its exact result (one f16
rounding an activation, test_gpu_qmm_tiles.py), so 8e-4 of the other; either
form of the delta rule 5e-6 (test_gpu_sparse.py), so 1e-5."""
import ctypes as C

import numpy as np
import pytest

from qwasar_amd import synth

pytestmark = pytest.mark.gpu


class qwk_q4(C.Structure):
    _fields_ = [("w", C.c_void_p), ("s", C.c_void_p), ("b", C.c_void_p)]


def rel_l2(a, b):
    a, b = np.asarray(a, np.float64).ravel(), np.asarray(b, np.float64).ravel()
    return float(np.sqrt(((a - b) ** 2).sum() / (b * b).sum()))


class Device:
    """Arrays in device memory, by the HIP runtime that the library links."""

    def __init__(self, gpu, **arrays):
        self.lib, self.arrays, self.at = C.CDLL(gpu.LIB_PATH), arrays, {}
        for name, a in arrays.items():
            a = np.ascontiguousarray(a)
            p = C.c_void_p()
            assert self.lib.hipMalloc(C.byref(p), C.c_size_t(a.nbytes)) == 0
            assert self.lib.hipMemcpy(p, C.c_void_p(a.ctypes.data), C.c_size_t(a.nbytes), 1) == 0
            self.at[name] = p

    def read(self, name):
        a = np.empty_like(self.arrays[name])
        assert self.lib.hipMemcpy(C.c_void_p(a.ctypes.data), self.at[name], C.c_size_t(a.nbytes), 2) == 0
        return a

    def bank(self):
        return qwk_q4(*[self.at[n].value for n in "wsb"])

    def call(self, name, *args):
        """qwk_<name> on the null stream, arrays by name; waits for it."""
        assert getattr(self.lib, name)(C.c_void_p(0), *[self.at[a] if isinstance(a, str) else a for a in args]) == 0
        assert self.lib.hipDeviceSynchronize() == 0

    def free(self):
        for p in self.at.values():
            assert self.lib.hipFree(p) == 0


def work_bytes(gpu, name, *args):
    f = getattr(C.CDLL(gpu.LIB_PATH), name)
    f.restype = C.c_size_t
    return f(*args)


@pytest.mark.parametrize("rows,k,n,G", [(16, 4096, 4100, 64), (67, 3072, 1024, 32), (200, 1152, 2000, 128),
                                        (8, 3072, 512, 64)])       # the last: small, split over k
def test_dense_product_without_scratch(gpu, rows, k, n, G):
    q = synth.make_q4(rows + n, "scratch", n, k, G)
    x = np.random.default_rng(rows).uniform(-1, 1, (rows, k)).astype(np.float32)
    assert work_bytes(gpu, "qwk_qmm_work_bytes", k, n, rows, G) > 0
    B = gpu.Buf
    wb, sb, bb, xb, yb = B.of(q.w), B.of(q.s), B.of(q.b), B.of(x), B(rows * n * 4)
    c = gpu.qw_cmd_begin()
    gpu.qw_op_qmm_q4(c, yb.ref(), xb.ref(), wb.ref(), sb.ref(), bb.ref(), k, n, rows, G)
    gpu.run(c, "qmm")
    dev = Device(gpu, w=q.w, s=q.s, b=q.b, x=x, y=np.full((rows, n), 7.0, np.float32))
    dev.call("qwk_qmm", "y", "x", dev.bank(), k, n, rows, G, None, C.c_size_t(0))
    assert rel_l2(dev.read("y"), yb.read(np.float32, (rows, n))) < 8e-4
    dev.free()


@pytest.mark.parametrize("E,K,rows,k,n,G,by_pair", [(64, 4, 33, 672, 200, 32, False), (16, 4, 61, 2560, 100, 64, False),
                                                    (8, 2, 130, 1152, 260, 128, True)])
def test_grouped_product_without_scratch(gpu, E, K, rows, k, n, G, by_pair):
    pairs = rows * K
    q = synth.make_q4(E + k, "scratch", E * n, k, G)
    g = np.random.default_rng(pairs)
    x = g.uniform(-1, 1, (pairs if by_pair else rows, k)).astype(np.float32)
    idx = np.stack([g.choice(E, K, replace=False) for _ in range(rows)]).astype(np.int32)
    B = gpu.Buf
    nt = gpu.qw_moe_max_tiles(pairs, E)
    wb, sb, bb, xb, ib = B.of(q.w), B.of(q.s), B.of(q.b), B.of(x), B.of(idx)
    perm, cur, tiles, yb = B(pairs * 4), B(E * 4), B((1 + 3 * nt) * 4), B(pairs * n * 4)
    c = gpu.qw_cmd_begin()
    gpu.qw_op_moe_group(c, perm.ref(), tiles.ref(), cur.ref(), ib.ref(), pairs, E)
    gpu.qw_op_qmm_q4_gather(c, yb.ref(), xb.ref(), perm.ref(), tiles.ref(), wb.ref(), sb.ref(), bb.ref(), k, n, pairs,
                            E, K, by_pair, G)
    gpu.run(c, "gather")
    tl, bm = tiles.read(np.int32, (1 + 3 * nt,)), gpu.qw_moe_tile_rows(pairs, E)
    assert 1 <= tl[0] <= nt and tl[3:3 + 3 * tl[0]:3].max() <= bm
    dev = Device(gpu, w=q.w, s=q.s, b=q.b, x=x, perm=perm.read(np.int32, (pairs,)), tiles=tl,
                 y=np.full((pairs, n), 7.0, np.float32))
    dev.call("qwk_gather_gemm", "y", "x", "perm", "tiles", dev.bank(), k, n, pairs, E, K, int(by_pair), G,
             bm, nt, None, C.c_size_t(0))
    assert rel_l2(dev.read("y"), yb.read(np.float32, (pairs, n))) < 8e-4
    dev.free()


def test_delta_rule_without_scratch(gpu):
    hk, hv, rows, d = 2, 4, 300, 128
    assert work_bytes(gpu, "qwk_gated_delta_work", hk, hv, rows, 0, 0) > 0
    g = np.random.default_rng(5)
    q, k = (g.standard_normal((rows, hk, d)).astype(np.float32) for _ in range(2))
    q /= np.linalg.norm(q, axis=-1, keepdims=True) * np.float32(np.sqrt(d))
    k /= np.linalg.norm(k, axis=-1, keepdims=True)
    v, s0 = g.uniform(-1, 1, (rows, hv, d)).astype(np.float32), g.uniform(-0.05, 0.05, (hv, d, d)).astype(np.float32)
    gate, beta = g.uniform(0.9, 0.99, (rows, hv)).astype(np.float32), g.uniform(0.3, 0.7, (rows, hv)).astype(np.float32)
    B = gpu.Buf
    qb, kb, vb, gb, bb, sb, yb = (B.of(a) for a in (q, k, v, gate, beta, s0, np.zeros_like(v)))
    c = gpu.qw_cmd_begin()
    gpu.qw_op_gated_delta(c, yb.ref(), qb.ref(), kb.ref(), vb.ref(), gb.ref(), bb.ref(), sb.ref(), hk, hv, d, d, rows,
                          gpu.NULL_REF, 0, 0)
    gpu.run(c, "gated delta")
    dev = Device(gpu, q=q, k=k, v=v, g=gate, beta=beta, s=s0, y=np.zeros_like(v))
    dev.call("qwk_gated_delta", "y", "q", "k", "v", "g", "beta", "s", hk, hv, d, d, rows, None, 0, 0, None, None)
    assert rel_l2(dev.read("y"), yb.read(np.float32, v.shape)) < 1e-5
    assert rel_l2(dev.read("s"), sb.read(np.float32, s0.shape)) < 1e-5
    dev.free()
