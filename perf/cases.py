"""The workloads that this library's speed is judged on: the sublayers of a
Flash-Next model as an engine drives them through the C ABI (qwasar_amd.gpu),
from one token to a 2048-token prefill chunk.

A pass is one command: qw_cmd_begin, the ops of one or more layers, then
qw_cmd_wait, the error check and qw_cmd_free (gpu.run).  Decode passes hold
several layers, because an engine encodes a token's layers into one command;
each layer has weights, caches and inputs of its own, so that every layer
reads its bytes from memory and a rounding difference in one layer does not
travel into the next.  Inputs are made by torch on the device from the seed
alone and copied into qw_bufs; buffers that stay on the device in an engine
(activations, states) are never exposed to the host.

Kinds of case:

  moe        qw_op_moe_layer over `layers` layers of `rows` tokens; with
             `residual`, qw_op_moe_layer_residual (the bf16 residual norm
             folded in); `route`: uniform, hot (three experts in every
             token's picks) or zipf router logits
  moe_ops    the same block op by op, as the reference's graph builder
             encodes it (qwasar_flash_graph.c:531-632)
  mixer      the hyper-connection mixer around a block: one launch a token,
             the op sequence for a chunk
  qsa        a sparse attention sublayer: stored block keys, block scores,
             selection, gated attention over the listed positions
  gdn        a gated DeltaNet sublayer: conv, delta rule, output gate
  proj       a dense 4-bit projection (qw_op_qmat_q4)
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from qwasar_amd import gpu

EPS = 1e-6
F64 = torch.float64
HOT = (7, 200, 411)          # the experts every token of a `hot` case picks
HOT_BIAS = 8.0               # their logits' lead
ZIPF_S = 1.1


# ---- the cases ----------------------------------------------------------------

def _moe(rows, layers=1, residual=False, route="uniform", H=3072, E=512, K=10, I=512, group=64, split=True):
    return {"kind": "moe", "rows": rows, "layers": layers, "residual": residual, "route": route, "H": H, "E": E,
            "K": K, "I": I, "group": group, "split": split}


def _moe_ops(rows, H, E, K, I, group, split):
    return {"kind": "moe_ops", "rows": rows, "layers": 1, "residual": False, "route": "uniform", "H": H, "E": E,
            "K": K, "I": I, "group": group, "split": split}


def _mixer(rows, layers, H=3072, lowrank=320, group=64):
    return {"kind": "mixer", "rows": rows, "layers": layers, "H": H, "S": 4, "lowrank": lowrank, "group": group}


def _qsa(rows, layers, ctx, topk=512):
    return {"kind": "qsa", "rows": rows, "layers": layers, "ctx": ctx, "topk": topk}


def _gdn(rows, layers, hk=16, hv=48):
    return {"kind": "gdn", "rows": rows, "layers": layers, "hk": hk, "hv": hv}


def _proj(rows, k, n, group=64):
    return {"kind": "proj", "rows": rows, "k": k, "n": n, "group": group}


def listed():
    return [
        # decoding one token: the MoE blocks of eight layers, the residual norm folded into each
        dict(_moe(1, layers=8, residual=True), name="moe_token"),
        # a verify batch of eight drafted tokens whose picks overlap
        dict(_moe(8, layers=4, route="hot"), name="moe_batch8"),
        # a 512-token prompt with the skewed expert load of natural text
        dict(_moe(512, route="zipf"), name="moe_prefill_zipf"),
        # one layer of a full 2048-token prefill chunk
        dict(_moe(2048, residual=True), name="moe_prefill_2048"),
        # a caller of the reference's op sequence, a ragged prompt, the released model's shape and
        # group 32 (its MLX export)
        dict(_moe_ops(301, 2560, 512, 10, 640, 32, True), name="moe_ops_prompt"),
        # decoding one token: the mixer of four layers, a few microseconds of device work each
        dict(_mixer(1, 4), name="mixer_token"),
        # the mixer over a ragged prompt
        dict(_mixer(1021, 1), name="mixer_prefill"),
        # decoding one token at the end of a 32K context, six sparse layers
        dict(_qsa(1, 6, 32768), name="qsa_token"),
        # a 512-token chunk at the end of a 16K context
        dict(_qsa(512, 1, 16384), name="qsa_prefill"),
        # decoding one token: twelve recurrent layers
        dict(_gdn(1, 12), name="gdn_token"),
        # a 2048-token chunk through one recurrent layer
        dict(_gdn(2048, 1), name="gdn_prefill"),
        # a recurrent layer's input projection over a 1024-token chunk
        dict(_proj(1024, 3072, 10240), name="proj_prefill"),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("moe", "moe", "moe_ops", "mixer", "qsa", "gdn", "proj"))
    if kind in ("moe", "moe_ops"):
        E = rng.choice((64, 128, 256, 512))
        group = rng.choice((32, 64, 128))
        g = max(group, 64)
        c = dict(H=64 * 2 * rng.randint(4, 24), E=E, K=rng.randint(4, 10), I=g * rng.randint(1, 640 // g),
                 group=group, split=rng.random() < 0.5)
        rows = _log(rng, 1, 1600)
        if kind == "moe_ops":
            return _moe_ops(rows, **c)
        return _moe(rows, layers=rng.randint(1, 8) if rows == 1 else rng.randint(1, 4) if rows <= 8 else 1,
                    residual=rng.random() < 0.5, **c)
    if kind == "mixer":
        rows = _log(rng, 1, 2048)
        return _mixer(rows, rng.randint(1, 12) if rows == 1 else 1, H=128 * rng.randint(8, 24),
                      lowrank=64 * rng.randint(2, 6), group=rng.choice((32, 64)))
    if kind == "qsa":
        rows = _log(rng, 1, 512)
        ctx = _log(rng, max(1024, 2 * rows), 32768 if rows == 1 else 16384)
        return _qsa(rows, rng.randint(1, 6) if rows == 1 else 1, ctx, topk=rng.choice((256, 512)))
    if kind == "gdn":
        rows = _log(rng, 1, 2048)
        hk = rng.choice((4, 8, 16))
        return _gdn(rows, rng.randint(1, 16) if rows == 1 else 1, hk=hk, hv=hk * rng.choice((2, 3)))
    return _proj(_log(rng, 1, 2048), 64 * rng.randint(16, 96), 64 * rng.randint(8, 160), group=rng.choice((32, 64)))


# ---- inputs ---------------------------------------------------------------------

class _Rand:
    """Seeded device tensors; every call draws on from one stream."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std

    def bf16(self, *shape, std=1.0):
        return self.normal(*shape, std=std).to(torch.bfloat16)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def words(self, *shape):
        return torch.randint(-2 ** 31, 2 ** 31, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def q4(self, rows, cols, group):
        """An MLX affine 4-bit matrix: uniform nibbles, scales U(0.001, 0.02), biases -8 * scale."""
        s = self.uniform(0.001, 0.02, rows, cols // group).to(torch.bfloat16)
        return self.words(rows, cols // 8), s, s * -8.0


def _router_bias(case, r):
    E = case["E"]
    if case["route"] == "hot":
        b = torch.zeros(E, device="cuda")
        b[torch.tensor(HOT, device="cuda")] = HOT_BIAS
        return b
    ranks = torch.randperm(E, generator=r.g, device="cuda").float() + 1.0
    return -ZIPF_S * torch.log(ranks)


def _moe_inputs(case, r):
    H, E, K, I, G, rows = (case[k] for k in ("H", "E", "K", "I", "group", "rows"))
    layers = []
    for _ in range(case["layers"]):
        t = {"router": r.bf16(E, H, std=0.02), "sh_gate_w": r.bf16(H, std=0.02)}
        for name, m, k in ((("gate", E * I, H), ("up", E * I, H)) if case["split"] else (("gate_up", 2 * E * I, H),)):
            t[name] = r.q4(m, k, G)
        t["down"] = r.q4(E * H, I, G)
        t["sh_gate"], t["sh_up"], t["sh_down"] = r.q4(I, H, G), r.q4(I, H, G), r.q4(H, I, G)
        if case["residual"]:
            t["h"], t["y_prev"] = r.bf16(rows, H), r.normal(rows, H)
        else:
            t["x"] = r.bf16(rows, H).float()
        if case["route"] != "uniform":
            # the expert's logit bias, through an input that is 1 in every row
            t["router"][:, 0] = _router_bias(case, r).to(torch.bfloat16)
            t["x"][:, 0] = 1.0
        layers.append(t)
    return layers


def _mixer_inputs(case, r):
    H, S, k, G, rows = (case[x] for x in ("H", "S", "lowrank", "group", "rows"))
    return [{"norm_w": r.uniform(0.9, 1.1, S * H).to(torch.bfloat16), "inj_w": r.bf16(S, S * H, std=0.02),
             "down": r.q4(k, S * H, G), "up": r.q4(S * H, k, G), "h4": r.normal(rows, S * H),
             "out": r.normal(rows, H), "inj": r.normal(rows, S)} for _ in range(case["layers"])]


# the indexer and the attention of the released model
RATIO, NQ, D_IDX, Q_HEADS, KV_HEADS, D_HEAD = 4, 16, 128, 24, 2, 256


def _qsa_inputs(case, r):
    rows, ctx, topk = case["rows"], case["ctx"], case["topk"]
    nb, base = (ctx + RATIO - 1) // RATIO, ctx - rows
    cap = gpu.qw_qsa_list_cap(topk, RATIO)
    layers = []
    for _ in range(case["layers"]):
        t = {"ikeys": r.normal(ctx, D_IDX), "k_norm": r.uniform(0.9, 1.1, D_IDX).to(torch.bfloat16),
             "inv_freq": (1e7 ** (-torch.arange(32, device="cuda", dtype=F64) / 32)).float(),
             "qn": r.normal(rows, NQ, D_IDX), "q": r.normal(rows, Q_HEADS, D_HEAD),
             "gate": r.normal(rows, Q_HEADS, D_HEAD),
             "k": r.normal(KV_HEADS, ctx, D_HEAD, std=0.5).half(), "v": r.normal(KV_HEADS, ctx, D_HEAD).half()}
        # the positions the attention reads: random blocks of each row's complete ones and the incomplete
        # tail, ascending, as a selection gives them.  Made here and not taken from this pass's selection, so
        # that a tie at the cut that rounding breaks does not hide what the attention's arithmetic gives.
        lst = torch.zeros(rows, 1 + cap, device="cuda", dtype=torch.int32)
        pick = torch.rand(rows, nb, generator=r.g, device="cuda")
        n = (base + torch.arange(rows, device="cuda") + 1) // RATIO
        pick[torch.arange(nb, device="cuda")[None, :] >= n[:, None]] = -1.0
        order = pick.argsort(dim=1, descending=True)[:, :topk]
        kk = order.shape[1]
        taken = n.clamp(max=topk)
        # a place past the row's complete blocks sorts to the end
        late = torch.arange(kk, device="cuda")[None, :] >= taken[:, None]
        blocks = order.masked_fill(late, nb + 1).sort(dim=1).values
        pos = torch.zeros(rows, cap, device="cuda", dtype=torch.long)
        pos[:, :kk * RATIO] = (blocks[:, :, None] * RATIO + torch.arange(RATIO, device="cuda")).flatten(1)
        tail = base + torch.arange(rows, device="cuda") + 1 - n * RATIO
        for j in range(RATIO - 1):
            rr = (j < tail).nonzero().flatten()
            pos[rr, taken[rr] * RATIO + j] = n[rr] * RATIO + j
        count = taken * RATIO + tail
        lst[:, 0] = count
        lst[:, 1:] = pos.masked_fill(torch.arange(cap, device="cuda")[None, :] >= count[:, None], 0)
        t["list"] = lst
        layers.append(t)
    return layers


def _gdn_inputs(case, r):
    hk, hv, rows = case["hk"], case["hv"], case["rows"]
    ch = (2 * hk + hv) * 128
    return [{"x": r.normal(rows, ch), "conv_w": r.bf16(ch, 4, std=0.3), "win": r.normal(3, ch),
             "a": r.normal(rows, hv), "b": r.normal(rows, hv),
             "A_log": torch.linspace(-0.5, 1.0, hv, device="cuda").to(torch.bfloat16),
             "dt_bias": torch.linspace(-0.2, 0.3, hv, device="cuda").to(torch.bfloat16),
             "S": r.normal(hv, 128, 128, std=0.05), "norm_w": r.uniform(0.9, 1.1, 128).to(torch.bfloat16),
             "z": r.normal(rows, hv, 128)} for _ in range(case["layers"])]


def _proj_inputs(case, r):
    return [{"x": r.normal(case["rows"], case["k"]), "w": r.q4(case["n"], case["k"], case["group"])}]


_INPUTS = {"moe": _moe_inputs, "moe_ops": _moe_inputs, "mixer": _mixer_inputs, "qsa": _qsa_inputs,
           "gdn": _gdn_inputs, "proj": _proj_inputs}


# ---- device buffers ---------------------------------------------------------------

class _Device:
    """A qw_buf's device memory as torch sees it.  The library exports no
    device address; it is the second field of a qw_buf (qwasar_hip.c,
    struct qw_buf_s), read here to hand inputs over and outputs back without
    a trip through the host.  Keeps the buffer alive."""

    _TYPES = {torch.float32: "<f4", torch.int32: "<i4", torch.uint8: "|u1", torch.float16: "<f2",
              torch.bfloat16: "<i2"}

    def __init__(self, buf, dtype, shape):
        self.buf = buf
        ptr = ctypes.cast(buf.handle, ctypes.POINTER(ctypes.c_void_p))[1]
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": self._TYPES[dtype],
                                         "data": (ptr, False), "version": 3}


def _view(buf, dtype, *shape):
    t = torch.as_tensor(_Device(buf, dtype, shape), device="cuda")
    return t.view(torch.bfloat16) if dtype == torch.bfloat16 else t


def _put(t):
    """A tensor's values in a qw_buf of its own."""
    b = gpu.Buf(t.numel() * t.element_size())
    _view(b, t.dtype, *t.shape).copy_(t)
    return b


def _f32(*shape):
    b = gpu.Buf(int(np.prod(shape)) * 4)
    return b, _view(b, torch.float32, *shape)


def _i32(*shape):
    b = gpu.Buf(int(np.prod(shape)) * 4)
    return b, _view(b, torch.int32, *shape)


class _Q4:
    def __init__(self, t, group):
        self.w, self.s, self.b = (_put(x) for x in t)
        self.group = group

    def refs(self):
        return self.w.ref(), self.s.ref(), self.b.ref()

    def q4(self):
        return gpu.qw_q4_ref(*self.refs(), self.group)


# ---- encoding: each builder gives a layer's ops and its outputs --------------------

def _moe_desc(case, t):
    """The layer's weights on the device and its descriptor."""
    G = case["group"]
    q = {n: _Q4(t[n], G) for n in ("gate_up", "gate", "up", "down", "sh_gate", "sh_up", "sh_down") if n in t}
    router, sgw = _put(t["router"]), _put(t["sh_gate_w"])
    none = gpu.qw_q4_ref(gpu.NULL_REF, gpu.NULL_REF, gpu.NULL_REF, 0)
    desc = gpu.qw_moe_layer(case["H"], case["E"], case["K"], case["I"], case["I"], True, case["split"], router.ref(),
                            *[q[n].q4() if n in q else none
                              for n in ("gate_up", "gate", "up", "down", "sh_gate", "sh_up", "sh_down")], sgw.ref())
    return desc, q, router, sgw


def _moe_build(case, t, keep):
    H, K, rows = case["H"], case["K"], case["rows"]
    desc, *bufs = _moe_desc(case, t)
    out, ov = _f32(rows, H)
    idx, iv = _i32(rows, K)
    w, wv = _f32(rows, K)
    keep += [desc, bufs]
    o = {"out": ov, "idx": iv, "w": wv}
    if not case["residual"]:
        x = _put(t["x"])
        keep.append(x)
        return [(gpu.qw_op_moe_layer, (out.ref(), idx.ref(), w.ref(), x.ref(), desc, rows))], o
    h, y, h2 = _put(t["h"]), _put(t["y_prev"]), gpu.Buf(rows * H * 2)
    x, xv = _f32(rows, H)
    keep += [h, y]
    o["h"], o["x"] = _view(h2, torch.bfloat16, rows, H), xv
    return [(gpu.qw_op_moe_layer_residual, (out.ref(), idx.ref(), w.ref(), h.ref(), y.ref(), h2.ref(), x.ref(), desc,
                                            rows, EPS))], o


def _moe_ops_build(case, t, keep):
    H, E, K, I, G, rows = (case[k] for k in ("H", "E", "K", "I", "group", "rows"))
    pairs = rows * K
    desc, q, router, sgw = _moe_desc(case, t)
    x = _put(t["x"])
    out, ov = _f32(rows, H)
    idx, iv = _i32(rows, K)
    w, wv = _f32(rows, K)
    logits, lv = _f32(rows, E)
    B = gpu.Buf
    sg, su, gs, sh = B(rows * I * 4), B(rows * I * 4), B(rows * 4), B(rows * H * 4)
    gu, act, y = B(pairs * 2 * I * 4), B(pairs * I * 4), B(pairs * H * 4)
    perm, cursor, tiles = B(pairs * 4), B(E * 4), B((1 + 3 * gpu.qw_moe_max_tiles(pairs, E)) * 4)
    keep += [desc, q, router, sgw, x, sg, su, gs, sh, gu, act, y, perm, cursor, tiles]
    X = x.ref()

    def dense(dst, src, name, k, n):
        return gpu.qw_op_qmat_q4, (dst.ref(), src.ref(), *q[name].refs(), k, n, rows, G)

    ops = [(gpu.qw_op_dmat_bf16, (logits.ref(), X, router.ref(), H, E, rows))]
    if rows == 1 and H >= 2048:
        parts = (gpu.qw_qmv_part * 2)(gpu.qw_qmv_part(sg.ref(), *q["sh_gate"].refs(), I),
                                      gpu.qw_qmv_part(su.ref(), *q["sh_up"].refs(), I))
        ops.append((gpu.qw_op_qmv_q4_multi, (X, H, G, 2, parts)))
    else:
        ops += [dense(sg, x, "sh_gate", H, I), dense(su, x, "sh_up", H, I)]
    ops += [(gpu.qw_op_dmat_bf16, (gs.ref(), X, sgw.ref(), H, 1, rows)),
            (gpu.qw_op_moe_route, (idx.ref(), w.ref(), logits.ref(), rows, E, K, True))]
    if rows == 1:
        shared = [(gpu.qw_op_qmv_q4_swiglu, (sh.ref(), sg.ref(), su.ref(), I, gpu.NULL_REF, *q["sh_down"].refs(), I,
                                             H, 1, G))]
    else:
        shared = [(gpu.qw_op_swiglu, (sg.ref(), sg.ref(), su.ref(), rows * I)), dense(sh, sg, "sh_down", I, H)]
    if rows > 8:          # the grouped products
        ops.append((gpu.qw_op_moe_group, (perm.ref(), tiles.ref(), cursor.ref(), idx.ref(), pairs, E)))

        def grouped(dst, src, name, k, n, by_pair):
            return gpu.qw_op_qmm_q4_gather, (dst, src, perm.ref(), tiles.ref(), *q[name].refs(), k, n, pairs, E, K,
                                             by_pair, G)

        if case["split"]:
            ops += [grouped(gu.ref(), X, "gate", H, I, False), grouped(gu.ref(pairs * I * 4), X, "up", H, I, False),
                    (gpu.qw_op_swiglu, (act.ref(), gu.ref(), gu.ref(pairs * I * 4), pairs * I))]
        else:
            ops += [grouped(gu.ref(), X, "gate_up", H, 2 * I, False),
                    (gpu.qw_op_swiglu_split, (act.ref(), gu.ref(), pairs, I))]
        ops += [grouped(y.ref(), act.ref(), "down", I, H, True)] + shared
    else:                 # a matvec a pair
        ops += shared
        if case["split"] and H >= 2048:
            ops.append((gpu.qw_op_qmv_q4_bank2, (gu.ref(), X, idx.ref(), *q["gate"].refs(), *q["up"].refs(), H, I,
                                                 pairs, K, G)))
        else:
            banks = (("gate", 0, I), ("up", pairs * I * 4, I)) if case["split"] else (("gate_up", 0, 2 * I),)
            ops += [(gpu.qw_op_qmv_q4_bank, (gu.ref(off), X, idx.ref(), *q[n].refs(), H, m, pairs, K, False, G))
                    for n, off, m in banks]
        up, stride = (pairs * I * 4, I) if case["split"] else (I * 4, 2 * I)
        ops.append((gpu.qw_op_qmv_q4_swiglu, (y.ref(), gu.ref(), gu.ref(up), stride, idx.ref(), *q["down"].refs(), I,
                                              H, pairs, G)))
    ops.append((gpu.qw_op_moe_combine_shared, (out.ref(), y.ref(), w.ref(), sh.ref(), gs.ref(), rows, K, H)))
    return ops, {"out": ov, "idx": iv, "w": wv, "logits": lv}


def _mixer_build(case, t, keep):
    H, S, k, G, rows = (case[x] for x in ("H", "S", "lowrank", "group", "rows"))
    HH = S * H
    nw, jw, dn, up = _put(t["norm_w"]), _put(t["inj_w"]), _Q4(t["down"], G), _Q4(t["up"], G)
    h4, out, inj = _put(t["h4"]), _put(t["out"]), _put(t["inj"])
    x, xv = _f32(rows, H)
    n4, nv = _f32(rows, HH)
    d, dv = _f32(rows, k)
    keep += [nw, jw, dn, up, h4, out, inj]
    if rows == 1:
        h2, hv = _f32(1, HH)
        j2, jv = _f32(1, S)
        return [(gpu.qw_op_hc_decode, (x.ref(), h2.ref(), n4.ref(), d.ref(), j2.ref(), h4.ref(), out.ref(), inj.ref(),
                                       nw.ref(), *dn.refs(), jw.ref(), *up.refs(), H, S, k, G, EPS, 1.0 / S))], \
            {"x": xv, "h4": hv, "n4": nv, "d": dv, "inj": jv}
    m = gpu.Buf(rows * HH * 4)
    keep.append(m)
    return [(gpu.qw_op_hc_inject_norm, (h4.ref(), out.ref(), inj.ref(), nw.ref(), n4.ref(), rows, H, S, EPS)),
            (gpu.qw_op_qmat_q4, (d.ref(), n4.ref(), *dn.refs(), HH, k, rows, G)),
            (gpu.qw_op_dmat_bf16, (inj.ref(), n4.ref(), jw.ref(), HH, S, rows)),
            (gpu.qw_op_silu_scale, (d.ref(), rows * k, 1.0 / S)),
            (gpu.qw_op_qmat_q4, (m.ref(), d.ref(), *up.refs(), k, HH, rows, G)),
            (gpu.qw_op_hc_mix, (x.ref(), n4.ref(), m.ref(), rows, H, S))], \
        {"x": xv, "h4": _view(h4, torch.float32, rows, HH), "n4": nv, "d": dv,
         "inj": _view(inj, torch.float32, rows, S)}


def _qsa_build(case, t, keep):
    rows, ctx, topk = case["rows"], case["ctx"], case["topk"]
    base, nb = ctx - rows, (ctx + RATIO - 1) // RATIO
    cap = gpu.qw_qsa_list_cap(topk, RATIO)
    b = {n: _put(v) for n, v in t.items()}
    pool, pv = _f32(nb, D_IDX)
    scores, sv = _f32(rows, nb)
    mask = gpu.Buf(rows * ctx)
    lst, lv = _i32(rows, 1 + cap)
    out, ov = _f32(rows, Q_HEADS, D_HEAD)
    keep += [b]
    # the blocks of the earlier positions have their keys in the pool already
    c = gpu.qw_cmd_begin()
    pool_args = (pool.ref(), b["ikeys"].ref(), b["k_norm"].ref(), b["inv_freq"].ref(), D_IDX, RATIO)
    torch.cuda.synchronize()
    gpu.qw_op_qsa_pool(c, *pool_args, 0, base // RATIO, 64, EPS)
    gpu.run(c, "qsa pool")
    ops = [(gpu.qw_op_qsa_pool, (*pool_args, base // RATIO, (base + rows) // RATIO, 64, EPS)),
           (gpu.qw_op_qsa_scores_pooled, (scores.ref(), b["qn"].ref(), pool.ref(), rows, NQ, D_IDX, RATIO, base, nb)),
           (gpu.qw_op_qsa_select, (mask.ref(), lst.ref(), scores.ref(), rows, RATIO, base, topk, ctx, nb)),
           (gpu.qw_op_attn_masked_gated, (out.ref(), b["gate"].ref(), b["q"].ref(), b["k"].ref(), b["v"].ref(),
                                          b["list"].ref(), rows, Q_HEADS, KV_HEADS, D_HEAD, ctx, base, 1.0 / 16.0,
                                          topk, RATIO))]
    return ops, {"out": ov, "scores": sv, "list": lv, "mask": _view(mask, torch.uint8, rows, ctx), "pool": pv}


def _gdn_build(case, t, keep):
    hk, hv, rows = case["hk"], case["hv"], case["rows"]
    kd, vd = hk * 128, hv * 128
    ch = 2 * kd + vd
    one = rows == 1
    S, cw, win = _put(t["S"]), t["conv_w"], t["win"]
    a, b, A, dt, nw, z = (_put(t[n]) for n in ("a", "b", "A_log", "dt_bias", "norm_w", "z"))
    prep = gpu.qw_gdn_prep(a.ref(), b.ref(), A.ref(), dt.ref(), EPS / 128, 1.0 / 128, 1.0 / math.sqrt(128))
    y = gpu.Buf(rows * vd * 4)
    o, ov = _f32(rows, hv, 128)
    keep += [S, a, b, A, dt, nw, z, prep, y]
    gate = (gpu.qw_op_rms_norm_gated_sigmoid, (o.ref(), y.ref(), nw.ref(), z.ref(), 128, rows * hv, EPS, 1.0))
    outs = {"out": ov, "y": _view(y, torch.float32, rows, hv, 128), "S": _view(S, torch.float32, hv, 128, 128)}
    if one:
        x, w, w0, w1 = _put(t["x"]), _put(cw), _put(win), gpu.Buf(3 * ch * 4)
        keep += [x, w, w0]
        outs["win"] = _view(w1, torch.float32, 3, ch)
        return [(gpu.qw_op_gdn_decode, (y.ref(), x.ref(), w0.ref(), w1.ref(), w.ref(), prep, S.ref(), hk, hv, 128,
                                        128)), gate], outs
    # a chunk: q, k and v from projections of their own, each through its channels' conv
    ops, mixed = [], []
    for name, lo, n in (("q", 0, kd), ("k", kd, kd), ("v", 2 * kd, vd)):
        x, w, wi = (_put(v.contiguous()) for v in (t["x"][:, lo:lo + n], cw[lo:lo + n], win[:, lo:lo + n]))
        m = gpu.Buf(rows * n * 4)
        keep += [x, w, wi, m]
        mixed.append(m)
        outs["win_" + name] = _view(wi, torch.float32, 3, n)
        ops.append((gpu.qw_op_conv1d_causal_silu, (m.ref(), x.ref(), wi.ref(), w.ref(), n, rows, 4, gpu.NULL_REF, 0,
                                                   0)))
    ops += [(gpu.qw_op_gated_delta_prep, (y.ref(), *[m.ref() for m in mixed], prep, S.ref(), hk, hv, 128, 128, rows,
                                          gpu.NULL_REF, 0, 0)), gate]
    return ops, outs


def _proj_build(case, t, keep):
    x, w = _put(t["x"]), _Q4(t["w"], case["group"])
    y, yv = _f32(case["rows"], case["n"])
    keep += [x, w]
    return [(gpu.qw_op_qmat_q4, (y.ref(), x.ref(), *w.refs(), case["k"], case["n"], case["rows"], case["group"]))], \
        {"y": yv}


_BUILD = {"moe": _moe_build, "moe_ops": _moe_ops_build, "mixer": _mixer_build, "qsa": _qsa_build, "gdn": _gdn_build,
          "proj": _proj_build}


def prepare(case, seed):
    gpu.init()
    layers = _INPUTS[case["kind"]](case, _Rand(seed))
    torch.cuda.synchronize()
    keep, ops, outs = [], [], []
    for t in layers:
        o, out = _BUILD[case["kind"]](case, t, keep)
        ops += o
        outs.append(out)
    torch.cuda.synchronize()
    return {"ops": ops, "outs": outs, "keep": keep}


def run(state):
    c = gpu.qw_cmd_begin()
    for op, args in state["ops"]:
        if op(c, *args) is False:
            raise RuntimeError(f"{op.__name__} refused")
    gpu.run(c, "pass")
    return state["outs"]


# ---- what a pass cannot do without ---------------------------------------------------

def _q4_bytes(rows, cols, group):
    return rows * cols // 2 + rows * (cols // group) * 4


def _unique_experts(case):
    """Experts that a layer's tokens are expected to pick between them."""
    E, K, rows = case["E"], case["K"], case["rows"]
    if case["route"] == "hot":
        return 3 + (E - 3) * (1 - (1 - (K - 3) / (E - 3)) ** rows)
    if case["route"] == "zipf":
        p = np.arange(1, E + 1) ** -ZIPF_S
        p = np.minimum(1.0, K * p / p.sum())
        return float((1 - (1 - p) ** rows).sum())
    return E * (1 - (1 - K / E) ** rows)


def work(case):
    kind, rows, L = case["kind"], case["rows"], case.get("layers", 1)
    if kind in ("moe", "moe_ops"):
        H, E, K, I, G = (case[k] for k in ("H", "E", "K", "I", "group"))
        expert = 2 * _q4_bytes(I, H, G) + _q4_bytes(H, I, G)
        b = (_unique_experts(case) + 1) * expert + 2 * E * H + 2 * H + rows * (2 * H * 4 + 2 * K * 4)
        b += rows * E * 4 if kind == "moe_ops" else rows * (2 * H * 2 + H * 4) if case["residual"] else 0
        f = rows * (2 * 3 * (K + 1) * I * H + 2 * E * H)
    elif kind == "mixer":
        H, S, k, G = (case[x] for x in ("H", "S", "lowrank", "group"))
        HH = S * H
        b = _q4_bytes(k, HH, G) + _q4_bytes(HH, k, G) + 2 * S * HH + 2 * HH
        b += rows * 4 * (3 * HH + 2 * H + k + 2 * S)
        f = rows * 2 * (2 * HH * k + HH * S)
    elif kind == "qsa":
        ctx, topk = case["ctx"], case["topk"]
        base, nb = ctx - rows, ctx // RATIO
        blocks = [(base + r + 1) // RATIO for r in range(rows)]
        listed_ = [min(topk, n) * RATIO + (base + r + 1) % RATIO for r, n in enumerate(blocks)]
        seen = min(ctx, sum(listed_))
        if rows > 1:     # positions that some row lists
            seen = ctx * (1 - math.prod(1 - min(1.0, x / (base + r + 1)) for r, x in enumerate(listed_)))
        b = nb * D_IDX * 4 + rows * (NQ * D_IDX + 3 * Q_HEADS * D_HEAD) * 4 + sum(blocks) * 4
        b += sum(base + r + 1 for r in range(rows)) + sum(4 * (1 + x) * 2 for x in listed_)
        b += 2 * KV_HEADS * seen * D_HEAD * 2 + RATIO * D_IDX * 4 * (rows // RATIO)
        f = 2.0 * NQ * D_IDX * sum(blocks) + 4.0 * Q_HEADS * D_HEAD * sum(listed_)
    elif kind == "gdn":
        hk, hv = case["hk"], case["hv"]
        ch = (2 * hk + hv) * 128
        b = 2 * hv * 128 * 128 * 4 + 2 * 3 * ch * 4 + ch * 8 + rows * 4 * (ch + 2 * hv + 3 * hv * 128)
        f = rows * (hv * 3 * 2 * 128 * 128 + ch * 8)
    else:
        k, n = case["k"], case["n"]
        b = _q4_bytes(n, k, case["group"]) + rows * (k + n) * 4
        f = 2.0 * rows * k * n
    return {"bytes": int(L * b), "flops": int(L * f)}


def tolerance(case):
    kind, rows = case["kind"], case["rows"]
    if kind == "moe" or (kind in ("moe_ops", "proj") and rows >= 8):
        # the products take their activations (on the matrix cores the dequantised weights too) as 16-bit
        # floats: 2 to 4e-4 from 64 bits.  Ids and the residual's bf16 carry come out the same.
        return {"rel": 1.5e-3, "max": 0.05, "differ": 1e-3}
    if kind == "mixer" and rows > 1:
        return {"rel": 1e-3, "max": 0.05}          # as above: 2.1e-4 on d
    if kind == "qsa":
        # 32-bit sums (the stored keys' rotation angle is a 32-bit product: 5e-5 from 64 bits on either side);
        # a block whose score ties at the cut may change places, and moves the rest of its row's list
        return {"rel": 1e-5, "max": 1e-3, "differ": 5e-3}
    return {"rel": 1e-5, "max": 1e-3}              # 32-bit sums: 1 to 5e-7 seen


# ---- the same in 64 bits ----------------------------------------------------------------

def _dequant(t, lo=0, n=None):
    """Rows lo .. lo + n of a 4-bit matrix."""
    w, s, b = (x[lo:lo + n] if n is not None else x for x in t)
    shift = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    q = ((w[:, :, None] >> shift) & 0xF).reshape(w.shape[0], -1).to(F64)
    g = q.shape[1] // s.shape[1]
    return q * s.to(F64).repeat_interleave(g, 1) + b.to(F64).repeat_interleave(g, 1)


def _silu(x):
    return x * torch.sigmoid(x)


def _rms(x, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _moe_exact(case, t):
    H, E, K, I = (case[k] for k in ("H", "E", "K", "I"))
    o = {}
    if case["residual"]:
        # the carry is bf16 by definition: one fp32 add, rounded
        h = (t["h"].float() + t["y_prev"]).to(torch.bfloat16)
        x = _rms(h.to(F64))
        o["h"], o["x"] = h, x
    else:
        x = t["x"].to(F64)
    logits = x @ t["router"].to(F64).T
    p = torch.softmax(logits, -1)
    w, idx = p.topk(K, dim=-1)
    w = w / w.sum(-1, keepdim=True)
    out = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        r, slot = (idx == e).nonzero(as_tuple=True)
        xe = x[r]
        if case["split"]:
            g, u = xe @ _dequant(t["gate"], e * I, I).T, xe @ _dequant(t["up"], e * I, I).T
        else:
            g, u = (xe @ _dequant(t["gate_up"], 2 * e * I, 2 * I).T).split(I, -1)
        out[r] += w[r, slot][:, None] * ((_silu(g) * u) @ _dequant(t["down"], e * H, H).T)
    sh = (_silu(x @ _dequant(t["sh_gate"]).T) * (x @ _dequant(t["sh_up"]).T)) @ _dequant(t["sh_down"]).T
    o["out"] = out + torch.sigmoid(x @ t["sh_gate_w"].to(F64))[:, None] * sh
    o["w"], o["idx"] = w, None
    if case["kind"] == "moe_ops":
        o["logits"] = logits
    return o


def _mixer_exact(case, t):
    H, S, rows = case["H"], case["S"], case["rows"]
    h4 = t["h4"].to(F64).view(rows, S, H)
    h4 = h4 + t["out"].to(F64)[:, None, :] * (2 * torch.sigmoid(t["inj"].to(F64) / S))[:, :, None]
    n4 = _rms(h4) * t["norm_w"].to(F64).view(S, H)
    flat = n4.view(rows, S * H)
    d = flat @ _dequant(t["down"]).T
    a = _silu(d / S)
    m = torch.sigmoid(a @ _dequant(t["up"]).T).view(rows, S, H)
    # a chunk's silu is in place, a token's down rows are kept as they are
    return {"x": (m * n4).mean(1), "h4": h4.view(rows, S * H), "n4": flat, "d": a if rows > 1 else d,
            "inj": flat @ t["inj_w"].to(F64).T}


def _qsa_exact(case, t):
    rows, ctx = case["rows"], case["ctx"]
    base, nb = ctx - rows, (ctx + RATIO - 1) // RATIO
    whole = ctx // RATIO
    key = _rms(t["ikeys"][:whole * RATIO].to(F64).view(whole, RATIO, D_IDX).mean(1)) * t["k_norm"].to(F64)
    ang = (torch.arange(whole, device="cuda", dtype=F64) * RATIO)[:, None] * t["inv_freq"].to(F64)
    c, s = ang.cos(), ang.sin()
    lo, hi = key[:, :32].clone(), key[:, 32:64].clone()
    key[:, :32], key[:, 32:64] = lo * c - hi * s, hi * c + lo * s
    scores = torch.zeros(rows, nb, device="cuda", dtype=F64)
    out = torch.empty(rows, Q_HEADS, D_HEAD, device="cuda", dtype=F64)
    G = Q_HEADS // KV_HEADS
    kc, vc = t["k"].to(F64), t["v"].to(F64)
    for lo_ in range(0, rows, 32):
        r = slice(lo_, min(lo_ + 32, rows))
        n = r.stop - r.start
        dots = t["qn"][r].to(F64).reshape(n * NQ, D_IDX) @ key.T
        sc = dots.clamp(min=0).view(n, NQ, whole).sum(1) / math.sqrt(D_IDX)
        nbr = (base + torch.arange(r.start, r.stop, device="cuda") + 1) // RATIO
        scores[r, :whole] = torch.where(torch.arange(whole, device="cuda")[None] < nbr[:, None], sc,
                                        torch.zeros_like(sc))
        lst = t["list"][r, 1:].long()
        dead = torch.arange(lst.shape[1], device="cuda")[None] >= t["list"][r, :1]
        q = t["q"][r].to(F64).view(n, KV_HEADS, G, D_HEAD)
        for h in range(KV_HEADS):
            k, v = kc[h][lst], vc[h][lst]                       # [n, cap, 256]
            z = torch.stack([q[i, h] @ k[i].T for i in range(n)]) / 16.0
            z = z.masked_fill(dead[:, None, :], -math.inf).softmax(-1)
            out[r, h * G:(h + 1) * G] = torch.stack([z[i] @ v[i] for i in range(n)])
    pool = torch.zeros(nb, D_IDX, device="cuda", dtype=F64)
    pool[:whole] = key
    return {"out": out * torch.sigmoid(t["gate"].to(F64)), "scores": scores, "list": None, "mask": None, "pool": pool}


def _gdn_exact(case, t):
    hk, hv, rows = case["hk"], case["hv"], case["rows"]
    kd, vd = hk * 128, hv * 128
    x = torch.cat((t["win"], t["x"])).to(F64)
    w = t["conv_w"].to(F64)
    m = _silu(sum(x[j:j + rows] * w[:, j] for j in range(4)))
    q, k, v = (u.reshape(rows, -1, 128) for u in m.split((kd, kd, vd), -1))
    q, k = _rms(q, EPS / 128) / 128, _rms(k, EPS / 128) / math.sqrt(128)
    q, k = q.repeat_interleave(hv // hk, 1), k.repeat_interleave(hv // hk, 1)
    sp = torch.nn.functional.softplus(t["a"].to(F64) + t["dt_bias"].to(F64))
    g, beta = torch.exp(-torch.exp(t["A_log"].to(F64)) * sp), torch.sigmoid(t["b"].to(F64))
    S = t["S"].to(F64)
    y = torch.empty(rows, hv, 128, device="cuda", dtype=F64)
    for i in range(rows):
        S = S * g[i, :, None, None]
        kv = (S * k[i, :, None, :]).sum(-1)
        S = S + ((v[i] - kv) * beta[i, :, None])[:, :, None] * k[i, :, None, :]
        y[i] = (S * q[i, :, None, :]).sum(-1)
    o = {"out": _rms(y) * t["norm_w"].to(F64) * torch.sigmoid(t["z"].to(F64)), "y": y, "S": S}
    win = x[rows:rows + 3]
    if rows == 1:
        o["win"] = win
    else:
        o["win_q"], o["win_k"], o["win_v"] = win[:, :kd], win[:, kd:2 * kd], win[:, 2 * kd:]
    return o


def _proj_exact(case, t):
    return {"y": t["x"].to(F64) @ _dequant(t["w"]).T}


_EXACT = {"moe": _moe_exact, "moe_ops": _moe_exact, "mixer": _mixer_exact, "qsa": _qsa_exact, "gdn": _gdn_exact,
          "proj": _proj_exact}


def exact(case, seed):
    return [_EXACT[case["kind"]](case, t) for t in _INPUTS[case["kind"]](case, _Rand(seed))]
