"""Timed cases of the fmt=6 int4 engine path: what a program that links libcoli_hip has it do.

A case is a dict of plain values; `path` names the entry points it goes through:

  gemv      coli_hip_gemv over S rows of x, all buffers on the device (a few rows: decode
            projections; S >= 4: the dense prefill GEMM)
  topk      coli_hip_gemv_topk: the lm_head of a decoded token with its 8 best logits
  moe       coli_hip_moe_decode: one layer's MoE block for one token
  prefill   coli_hip_moe_prefill: one layer's MoE block over the S rows of a prompt
  experts   the engine's own prefill MoE calls on host buffers: coli_vk_eg_xs_bind, one
            coli_vk_expert_group_issue_id / _take per chunk of <= 64 experts and <= 1024 rows,
            the shared expert over all rows
  gqa       coli_vk_gqa_full over S rows on host buffers: a gated attention layer of a prompt
  gdn       coli_vk_gdn_full_seq over S rows on host buffers: a GatedDeltaNet layer of a prompt
  layers    coli_vk_stream_begin, the *_full_route_pipe blocks of four layers (three
            GatedDeltaNet, one attention, the MoE of each fused), coli_vk_stream_end: a tenth
            of one decoded token of the 40-layer model

Sizes are those of the model the benchmark builds (D 2048, 256 experts of width 512, top 8,
16 query / 2 key-value heads of 256, 32 value heads of 128, vocabulary 248320, group size
128) and, in draws, sizes around them.  Weights are round-to-nearest int4 codes of normal
weights (codes around their real-valued zero point), x is normed activations with a few
large channels.
"""
import ctypes
import importlib.util
import math
import os

import numpy as np
import torch

GS = 128
D, I, E, K = 2048, 512, 256, 8
H, KH, HD, ROT, MAX_T, THETA = 16, 2, 256, 64, 4096, 1e7
GKH, GKD, GVH, GVD, GCK = 16, 128, 32, 128, 4
GCD = 2 * GKH * GKD + GVH * GVD
EPS = 1e-6
VOCAB = 248320
MAX_EXPERTS, MAX_ROWS = 64, 1024   # of one expert-group call, as the engine chunks them
F64 = torch.float64


def listed():
    return [
        # one projection (the attention block's query | gate rows) of two tokens, a draft and
        # the one before it: the smallest call, bound by its launches
        {"name": "gemv_8192x2048_s2", "path": "gemv", "O": 8192, "I": 2048, "S": 2},
        # the qkv projection of a 512-row prompt piece
        {"name": "gemm_8192x2048_s512", "path": "gemv", "O": 8192, "I": 2048, "S": 512},
        # the output projection of a short, odd prompt (its rows fill no tile evenly)
        {"name": "gemm_2048x4096_s45", "path": "gemv", "O": 2048, "I": 4096, "S": 45},
        # the lm_head of every decoded token
        {"name": "lm_head_top8", "path": "topk", "O": VOCAB, "I": 2048, "k": 8},
        # a layer's MoE block of one decoded token
        {"name": "moe_decode", "path": "moe", "E": E, "K": K, "D": D, "I": I, "router": "f32"},
        # the MoE block of a short chat turn: most experts get a row or none; int8 router
        {"name": "moe_prefill_s37", "path": "prefill", "S": 37, "E": E, "K": K, "D": D, "I": I, "router": "int8"},
        # of an ordinary prompt
        {"name": "moe_prefill_s512", "path": "prefill", "S": 512, "E": E, "K": K, "D": D, "I": I, "router": "f32"},
        # of a long prompt
        {"name": "moe_prefill_s2000", "path": "prefill", "S": 2000, "E": E, "K": K, "D": D, "I": I, "router": "f32"},
        # the unchanged engine's expert-group calls for a 256-row prompt, host buffers both ways
        {"name": "experts_s256", "path": "experts", "S": 256},
        # an attention layer over a long prompt
        {"name": "gqa_s1900", "path": "gqa", "S": 1900, "pos": 0},
        # a GatedDeltaNet layer over a prompt that ends inside a chunk
        {"name": "gdn_s777", "path": "gdn", "S": 777},
        # four layers of a decoded token near the end of a 4096-row cache
        {"name": "layers_pos4000", "path": "layers", "pos": 4000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["gemv", "gemv", "gemv", "topk", "moe", "prefill", "prefill", "prefill", "experts", "gqa",
                       "gqa", "gdn", "gdn", "layers"])
    if path == "gemv":
        return {"path": path, "O": _log_int(rng, 256, 12288), "I": GS * rng.randint(4, 32),
                "S": rng.choice([rng.randint(2, 4), _log_int(rng, 4, 64), _log_int(rng, 64, 512)])}
    if path == "topk":
        return {"path": path, "O": _log_int(rng, 32000, VOCAB), "I": GS * rng.randint(8, 16), "k": rng.randint(1, 8)}
    if path in ("moe", "prefill"):
        c = {"path": path, "E": rng.choice([64, 128, 256]), "K": rng.choice([4, 6, 8]), "D": rng.choice([1024, 2048]),
             "I": rng.choice([256, 512]), "router": rng.choice(["f32", "int8"])}
        if path == "prefill":
            c["S"] = _log_int(rng, 2, 2000)
        return c
    if path == "experts":
        return {"path": path, "S": _log_int(rng, 8, 256)}
    if path == "gqa":
        S = _log_int(rng, 4, 1900)
        return {"path": path, "S": S, "pos": rng.choice([0, rng.randint(1, max(1, 1900 - S))])}
    if path == "gdn":
        return {"path": path, "S": _log_int(rng, 4, 1500)}
    return {"path": path, "pos": _log_int(rng, 1, MAX_T - 1)}


# ---------------------------------------------------------------- seeded inputs
def _gen(seed, *tags):
    h = 1469598103934665603
    for v in (seed, *tags):
        h = ((h ^ (int(v) & 0xFFFFFFFF)) * 1099511628211) & 0x7FFFFFFFFFFFFFFF
    return torch.Generator(device="cuda").manual_seed(h)


def _normal(shape, sigma, seed, *tags):
    return torch.randn(shape, device="cuda", generator=_gen(seed, *tags)) * sigma


def _acts(rows, n, seed, tag):
    """Normed activations: unit normal, one channel in 100 eight times as large."""
    big = 1.0 + 7.0 * (torch.rand(n, device="cuda", generator=_gen(seed, tag, 1)) < 0.01).float()
    return _normal((rows, n), 1.0, seed, tag) * big


def _int4(n, out_f, in_f, seed, tag):
    """n matrices [out_f, in_f] of int4 codes, two a byte (even column low), and their
    [scale, zero] pairs per group: weights of deviation about 0.02."""
    ng = in_f // GS
    q = torch.empty((n, out_f, in_f // 2), dtype=torch.uint8, device="cuda")
    g = _gen(seed, tag)
    step = max(1, (1 << 26) // (out_f * in_f))
    for a in range(0, n, step):
        b = min(n, a + step)
        c = (torch.randn((b - a, out_f, in_f), device="cuda", generator=g) * 2.6 + 7.5).round_().clamp_(0, 15)
        c = c.to(torch.uint8)
        q[a:b] = c[..., 0::2] | (c[..., 1::2] << 4)
    sz = torch.empty((n, out_f, ng, 2), device="cuda")
    sz[..., 0] = (0.0077 * (1.0 + 0.3 * torch.rand((n, out_f, ng), device="cuda", generator=g))).half().float()
    sz[..., 1] = 7.5 + 0.5 * torch.randn((n, out_f, ng), device="cuda", generator=g)
    return q, sz


def _int8(out_f, in_f, seed, tag):
    """Rows of int8 codes and their scales: the engine's router and GatedDeltaNet a / b."""
    w = _normal((out_f, in_f), 0.02, seed, tag)
    s = w.abs().amax(1) / 127.0
    return (w / s[:, None]).round().clamp(-127, 127).to(torch.int8), s


def _wide4(q, sz):
    """The int4 matrices in 64 bits."""
    c = torch.stack((q & 15, q >> 4), -1).reshape(*q.shape[:-1], -1).to(F64)
    c = c.reshape(*c.shape[:-1], -1, GS)
    s = sz.to(F64)
    return ((c - s[..., 1:2]) * s[..., 0:1]).reshape(*q.shape[:-1], -1)


def _wide8(q, s):
    return q.to(F64) * s.to(F64)[:, None]


# ---------------------------------------------------------------- the library
_lib = None


def _library():
    global _lib
    if _lib is None:
        here = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen3.c_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location("qwen3_c_amd", here)
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        _lib = mod.Lib().init()
    return _lib


class _Slots:
    """Indexes of the library's per-layer state, given back when the case's state goes."""

    def __init__(self, free):
        self.free = list(free)

    def take(self, n):
        got, self.free = self.free[:n], self.free[n:]
        if len(got) < n:
            raise RuntimeError("no layer index left")
        return got


class _Lease:
    def __init__(self, slots, n):
        self.slots, self.ids = slots, slots.take(n)

    def __del__(self):
        self.slots.free.extend(self.ids)


TABLE_LAYERS = 40
_table = {"dims": None, "slots": None}
_kv, _gdn = _Slots(range(160)), _Slots(range(160))   # one shape each: an index keeps its first


def _table_slots(dims):
    if _table["dims"] != dims:
        e, d, i = dims
        _library().eg_table_init(TABLE_LAYERS, e, d, i, GS)
        _table["dims"], _table["slots"] = dims, _Slots(range(TABLE_LAYERS))
    return _table["slots"]


def _up4(q, sz):
    """Uploads [n] int4 matrices; returns the tensors."""
    lib, qh, sh = _library(), q.cpu().numpy(), sz.cpu().numpy()
    return [lib.tensor(qh[i], sh[i], 6, qh.shape[2] * 2, qh.shape[1], GS) for i in range(qh.shape[0])]


def _up1(q, sz):
    return _up4(q, sz)[0]


def _up8(q, s):
    return _library().tensor(q.cpu().numpy().view(np.uint8), s.cpu().numpy(), 1, q.shape[1], q.shape[0])


def _experts(e, d, i, seed, tag):
    """Gate, up [e + 1, i, d] and down [e + 1, d, i] of a layer (the shared expert last), the
    shared expert's gate vector."""
    return (_int4(e + 1, i, d, seed, tag), _int4(e + 1, i, d, seed, tag + 1), _int4(e + 1, d, i, seed, tag + 2),
            _normal(d, 0.02, seed, tag + 3))


def _router(e, d, kind, seed, tag):
    """(uploaded tensor maker, 64-bit rows) of a router."""
    if kind == "int8":
        q, s = _int8(e, d, seed, tag)
        return lambda: _up8(q, s), lambda: _wide8(q, s)
    w = _normal((e, d), 0.02, seed, tag)
    return lambda: _library().tensor(w.cpu().numpy(), None, 0, d, e), lambda: w.to(F64)


def _put_table(layer, ex):
    lib = _library()
    g, u, dn = _up4(*ex[0]), _up4(*ex[1]), _up4(*ex[2])
    n = len(g) - 1
    for e in range(n):
        lib.eg_table_set(layer, e, g[e], u[e], dn[e])
    lib.eg_table_set_shared(layer, g[n], u[n], dn[n], ex[3].cpu().numpy())
    return g, u, dn


def _host(t):
    return np.ascontiguousarray(t.cpu().numpy())


# ---------------------------------------------------------------- cases
def _gqa_weights(seed, tag):
    return {"q": _int4(1, 2 * H * HD, D, seed, tag), "k": _int4(1, KH * HD, D, seed, tag + 1),
            "v": _int4(1, KH * HD, D, seed, tag + 2), "o": _int4(1, D, H * HD, seed, tag + 3),
            "qn": _normal(HD, 0.1, seed, tag + 4), "kn": _normal(HD, 0.1, seed, tag + 5)}


def _gdn_weights(seed, tag):
    return {"qkv": _int4(1, GCD, D, seed, tag), "z": _int4(1, GVH * GVD, D, seed, tag + 1),
            "out": _int4(1, D, GVH * GVD, seed, tag + 2), "conv": _normal((GCD, GCK), 0.3, seed, tag + 3),
            "alog": _normal(GVH, 0.5, seed, tag + 4), "dtb": _normal(GVH, 1.0, seed, tag + 5),
            "gnorm": 1.0 + _normal(GVD, 0.1, seed, tag + 6), "a": _int8(GVH, D, seed, tag + 7),
            "b": _int8(GVH, D, seed, tag + 8)}


def _gdn_params(w, x):
    """[decay | beta | norm weight] per row, as the engine packs them."""
    a = x.to(F64) @ _wide8(*w["a"]).T + w["dtb"].to(F64)
    b = x.to(F64) @ _wide8(*w["b"]).T
    decay = torch.exp(-torch.exp(w["alog"].to(F64)) * torch.nn.functional.softplus(a))
    return torch.cat((decay, torch.sigmoid(b), w["gnorm"].to(F64).expand(x.shape[0], GVD)), 1).float().contiguous()


def _cache(seed, tag, n):
    """Keys (normed, of about unit size) and values of n earlier positions [KH, n, HD]."""
    return _normal((KH, n, HD), 1.0, seed, tag), _normal((KH, n, HD), 1.0, seed, tag + 1)


def _load_cache(layer, kc, vc):
    lib, n = _library(), kc.shape[1]
    lib.kv_ensure(layer, KH * MAX_T, HD, HD)
    if n:
        kh, vh = _host(kc), _host(vc)
        for h in range(KH):
            lib.kv_load(layer, h * MAX_T, kh[h], vh[h])


def _route_ids(s, seed, tag):
    """Top K of E experts per row, some experts more popular than others, and ids in rank order."""
    lg = _normal((s, E), 1.0, seed, tag) + _normal(E, 0.5, seed, tag + 1)
    return lg.topk(K, dim=1).indices.cpu().numpy()


def _chunks(ids):
    """The (experts, rows, token ids) of the engine's expert-group calls."""
    flat = ids.reshape(-1)
    order = np.argsort(flat, kind="stable")
    out, cur, n = [], [], 0
    ends = np.searchsorted(flat[order], np.arange(E + 1))
    for e in range(E):
        a = int(ends[e])
        while a < ends[e + 1]:
            if len(cur) == MAX_EXPERTS or n == MAX_ROWS:
                out.append(cur)
                cur, n = [], 0
            b = min(int(ends[e + 1]), a + MAX_ROWS - n)
            cur.append((e, order[a:b] // K))
            n += b - a
            a = b
    out.append(cur)
    return out


def prepare(case, seed):
    lib, p = _library(), case["path"]
    st = {"path": p}
    if p == "gemv":
        st["t"] = _up1(*_int4(1, case["O"], case["I"], seed, 1))
        st["x"] = _acts(case["S"], case["I"], seed, 2)
        st["y"] = torch.empty((case["S"], case["O"]), device="cuda")
    elif p == "topk":
        st["t"], st["k"] = _up1(*_int4(1, case["O"], case["I"], seed, 1)), case["k"]
        st["x"] = _acts(1, case["I"], seed, 2)
        st["y"] = torch.empty(case["O"], device="cuda")
        st["idx"] = torch.empty(case["k"], dtype=torch.int32, device="cuda")
        st["val"] = torch.empty(case["k"], device="cuda")
    elif p in ("moe", "prefill"):
        d, k, s = case["D"], case["K"], case.get("S", 1)
        st["lease"] = _Lease(_table_slots((case["E"], d, case["I"])), 1)
        st["layer"], st["K"], st["S"] = st["lease"].ids[0], k, s
        st["keep"] = _put_table(st["layer"], _experts(case["E"], d, case["I"], seed, 10))
        st["router"] = _router(case["E"], d, case["router"], seed, 3)[0]()
        st["x"] = _acts(s, d, seed, 2)
        st["out"] = torch.empty((s, d), device="cuda")
        st["idx"] = torch.empty((s, k), dtype=torch.int32, device="cuda")
        st["val"] = torch.empty((s, k) if p == "prefill" else k + 1, device="cuda")
    elif p == "experts":
        s = case["S"]
        g, u, dn, _ = _experts(E, D, I, seed, 10)
        g, u, dn = _up4(*g), _up4(*u), _up4(*dn)
        st["keep"], st["S"], st["x"] = (g, u, dn), s, _host(_acts(s, D, seed, 2))
        st["calls"], at = [], 0
        st["y"] = np.zeros((s * K + s, D), np.float32)
        arr = lambda ts, es: (ctypes.c_void_p * len(es))(*[ts[e].handle.value for e in es])  # noqa: E731
        for ch in _chunks(_route_ids(s, seed, 4)):
            es, tok = [c[0] for c in ch], np.ascontiguousarray(np.concatenate([c[1] for c in ch]), np.int32)
            rows = (ctypes.c_int * len(es))(*[len(c[1]) for c in ch])
            st["calls"].append((arr(g, es), arr(u, es), arr(dn, es), rows, len(es), tok, st["y"][at:at + len(tok)]))
            at += len(tok)
        st["shared"] = (arr(g, [E]), arr(u, [E]), arr(dn, [E]), (ctypes.c_int * 1)(s), 1, st["y"][at:])
    elif p == "gqa":
        w = _gqa_weights(seed, 20)
        st["lease"] = _Lease(_kv, 1)
        st["layer"], st["S"], st["pos"] = st["lease"].ids[0], case["S"], case["pos"]
        st["t"] = [_up1(*w[n]) for n in ("q", "k", "v", "o")]
        _load_cache(st["layer"], *_cache(seed, 40, case["pos"]))
        lib.gqa_norm_weight(st["layer"], _host(w["qn"]), _host(w["kn"]))
        st["x"] = _host(_acts(case["S"], D, seed, 2))
    elif p == "gdn":
        w = _gdn_weights(seed, 20)
        st["lease"] = _Lease(_gdn, 1)
        st["layer"], st["S"] = st["lease"].ids[0], case["S"]
        st["t"] = [_up1(*w[n]) for n in ("qkv", "z", "out")]
        x = _acts(case["S"], D, seed, 2)
        lib.gdn_setup(st["layer"], GVH, GKD, GVD, GCK, GCD, _host(w["conv"].reshape(-1)))
        lib.gdn_reset()   # a new sequence
        st["x"], st["params"] = _host(x), _host(_gdn_params(w, x))
    else:
        st["pos"], st["layers"] = case["pos"], []
        st["lease"] = [_Lease(_table_slots((E, D, I)), 4), _Lease(_kv, 1), _Lease(_gdn, 3)]
        slots, kv, gd = (x.ids for x in st["lease"])
        for n in range(4):
            tag = 100 * (n + 1)
            w = _gqa_weights(seed, tag) if n == 3 else _gdn_weights(seed, tag)
            keep = _put_table(slots[n], _experts(E, D, I, seed, tag + 50))
            router = _router(E, D, "int8", seed, tag + 60)[0]()
            lib.layer_norm_weight(slots[n], _host(_normal(D, 0.1, seed, tag + 61)), _host(_normal(D, 0.1, seed, tag + 62)))
            if n == 3:
                t = [_up1(*w[m]) for m in ("q", "k", "v", "o")]
                _load_cache(kv[0], *_cache(seed, 40, case["pos"]))
                lib.gqa_norm_weight(kv[0], _host(w["qn"]), _host(w["kn"]))
            else:
                t = [_up1(*w["qkv"]), _up1(*w["z"]), _up8(*w["a"]), _up8(*w["b"]), _up1(*w["out"])]
                lib.gdn_setup(gd[n], GVH, GKD, GVD, GCK, GCD, _host(w["conv"].reshape(-1)), _host(w["alog"]),
                              _host(w["dtb"]), _host(w["gnorm"]))
            st["layers"].append((kv[0] if n == 3 else gd[n], t, router, slots[n], keep))
        lib.gdn_reset()
        st["x"] = _host(_normal(D, 1.0, seed, 2))
    return st


def run(st):
    lib, p = _library(), st["path"]
    if p == "gemv":
        lib.gemv_dev(st["t"], st["x"].data_ptr(), st["y"].data_ptr(), st["x"].shape[0])
        return st["y"]
    if p == "topk":
        lib.gemv_topk_dev(st["t"], st["x"].data_ptr(), st["y"].data_ptr(), st["k"], st["idx"].data_ptr(),
                          st["val"].data_ptr())
        return st["y"], st["val"], st["idx"]
    if p == "moe":
        lib.moe_decode_dev(st["layer"], st["router"], st["K"], st["x"].data_ptr(), st["out"].data_ptr(), False,
                           st["idx"].data_ptr(), st["val"].data_ptr())
        return st["out"], st["val"], st["idx"]
    if p == "prefill":
        lib.moe_prefill_dev(st["layer"], st["router"], st["K"], st["x"].data_ptr(), st["S"], st["out"].data_ptr(),
                            st["idx"].data_ptr(), st["val"].data_ptr())
        return st["out"], st["val"], st["idx"]
    if p == "experts":
        ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
        lib.eg_xs_bind(st["x"], st["S"], D)
        for g, u, dn, rows, n, tok, y in st["calls"]:
            if not lib.L.coli_vk_expert_group_issue_id(g, u, dn, rows, n, ptr(tok)):
                raise RuntimeError("coli_vk_expert_group_issue_id")
            lib.expert_group_take_into(y)
        g, u, dn, rows, n, y = st["shared"]
        if not lib.L.coli_vk_expert_group_issue(g, u, dn, rows, n, ptr(st["x"])):
            raise RuntimeError("coli_vk_expert_group_issue")
        lib.expert_group_take_into(y)
        return st["y"]
    if p == "gqa":
        return lib.gqa_full(st["layer"], st["x"], *st["t"], st["S"], H, KH, HD, ROT, st["pos"], MAX_T, EPS, THETA)
    if p == "gdn":
        return lib.gdn_full_seq(st["layer"], st["x"], st["params"], *st["t"], st["S"], GKH, GKD, GVH, GVD, GCD, GCK, EPS)
    lib.stream_begin(st["x"])
    for n, (idx, t, router, slot, _) in enumerate(st["layers"]):
        if n == 3:
            lib.gqa_route_pipe(idx, *t, router, slot, K, H, KH, HD, ROT, st["pos"], MAX_T, EPS, THETA)
        else:
            lib.gdn_route_pipe(idx, *t, router, slot, K, GKH, GKD, GVH, GVD, GCD, GCK, EPS)
    return lib.stream_end(D)


# ---------------------------------------------------------------- what a pass cannot do without
def _b4(out_f, in_f):
    return out_f * in_f // 2 + out_f * (in_f // GS) * 8


def _expert_bytes(d, i):
    return 2 * _b4(i, d) + _b4(d, i)


def _moe_work(s, c, touched):
    d, i, e, k = c["D"], c["I"], c["E"], c["K"]
    rb = e * d * (1 if c["router"] == "int8" else 4)
    return (touched + 1) * _expert_bytes(d, i) + rb + d * 4 + 2 * s * d * 4, 6 * s * (k + 1) * d * i + 2 * s * (e + 1) * d


def work(case):
    p = case["path"]
    if p == "gemv":
        o, i, s = case["O"], case["I"], case["S"]
        return {"bytes": _b4(o, i) + 4 * s * (i + o), "flops": 2 * s * o * i}
    if p == "topk":
        return {"bytes": _b4(case["O"], case["I"]) + 4 * (case["I"] + case["O"]), "flops": 2 * case["O"] * case["I"]}
    if p in ("moe", "prefill"):
        s = case.get("S", 1)
        touched = case["E"] * (1 - (1 - case["K"] / case["E"]) ** s)   # experts that s rows reach
        b, f = _moe_work(s, case, touched)
        return {"bytes": b, "flops": f}
    if p == "experts":
        s = case["S"]
        touched = E * (1 - (1 - K / E) ** s)
        return {"bytes": (touched + 1) * _expert_bytes(D, I) + 4 * s * D * (K + 3), "flops": 6 * s * (K + 1) * D * I}
    if p == "gqa":
        s, n = case["S"], case["S"] * case["pos"] + case["S"] * (case["S"] + 1) // 2   # query-key pairs
        wts = _b4(2 * H * HD, D) + 2 * _b4(KH * HD, D) + _b4(D, H * HD)
        return {"bytes": wts + 8 * s * D + 8 * KH * HD * (case["pos"] + 2 * s),
                "flops": 2 * s * D * (3 * H * HD + 2 * KH * HD) + 4 * n * H * HD}
    if p == "gdn":
        s = case["S"]
        wts = _b4(GCD, D) + _b4(GVH * GVD, D) + _b4(D, GVH * GVD)
        state = 4 * (GVH * GKD * GVD + GCK * GCD)
        return {"bytes": wts + 2 * state + 4 * s * (2 * D + 2 * GVH + GVD),
                "flops": 2 * s * D * (GCD + 2 * GVH * GVD) + 7 * s * GVH * GKD * GVD}
    b, f = _moe_work(1, {"D": D, "I": I, "E": E, "K": K, "router": "int8"}, K)
    gdn = (_b4(GCD, D) + 2 * _b4(GVH * GVD, D) + 2 * GVH * (D + 4) + 8 * (GVH * GKD * GVD + GCK * GCD),
           2 * D * (GCD + 2 * GVH * GVD + 2 * GVH) + 7 * GVH * GKD * GVD)
    gqa = (_b4(2 * H * HD, D) + 2 * _b4(KH * HD, D) + _b4(D, H * HD) + 8 * KH * HD * (case["pos"] + 1),
           2 * D * (3 * H * HD + 2 * KH * HD) + 4 * (case["pos"] + 1) * H * HD)
    return {"bytes": 4 * b + 3 * gdn[0] + gqa[0], "flops": 4 * f + 3 * gdn[1] + gqa[1]}


def tolerance(case):
    """32-bit results from exact integer products: four times what another order of the sums
    shows against 64 bits.  The recurrence and the four layers carry a rounding on."""
    return {"gemv": {"rel": 4e-6}, "topk": {"rel": 4e-6, "differ": 0.001}, "moe": {"rel": 4e-6, "differ": 0.001},
            "prefill": {"rel": 4e-6, "differ": 0.001}, "experts": {"rel": 4e-6}, "gqa": {"rel": 1e-5},
            "gdn": {"rel": 1e-5}, "layers": {"rel": 1e-5}}[case["path"]]


# ---------------------------------------------------------------- the same in 64 bits
def _mlp(x, ex, e):
    g, u = x @ _wide4(ex[0][0][e], ex[0][1][e]).T, x @ _wide4(ex[1][0][e], ex[1][1][e]).T
    return (torch.nn.functional.silu(g) * u) @ _wide4(ex[2][0][e], ex[2][1][e]).T


def _moe64(x, router, ex, k):
    """(out, weights, ids, shared gate) of rows x."""
    p = torch.softmax(x @ router.T, 1)
    v, ids = p.topk(k, dim=1)
    v = v / v.sum(1, keepdim=True)
    sh = torch.sigmoid(x @ ex[3].to(F64))
    out = sh[:, None] * _mlp(x, ex, ex[0][0].shape[0] - 1)
    for e in ids.unique().tolist():
        r, c = (ids == e).nonzero(as_tuple=True)
        out.index_add_(0, r, _mlp(x[r], ex, e) * v[r, c][:, None])
    return out, v, ids, sh


def _norm64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * (1.0 + w.to(F64))


def _rope64(x, pos):
    """Rows x [s, heads, HD] at positions pos .. ; the angles are the path's 32-bit products."""
    hr = ROT // 2
    inv = np.array([np.float32(float(np.float32(THETA)) ** float(np.float32(-2.0 * j / ROT))) for j in range(hr)], np.float32)
    ang = (np.arange(pos, pos + x.shape[0], dtype=np.float32)[:, None] * inv[None]).astype(np.float64)
    cs, sn = (torch.from_numpy(f(ang)).cuda()[:, None] for f in (np.cos, np.sin))
    lo, hi = x[..., :hr], x[..., hr:ROT]
    return torch.cat((lo * cs - hi * sn, hi * cs + lo * sn, x[..., ROT:]), -1)


def _gqa64(x, w, kc, vc):
    s, pos = x.shape[0], kc.shape[1]
    qg = (x @ _wide4(*w["q"])[0].T).reshape(s, H, 2 * HD)
    q, gate = _rope64(_norm64(qg[..., :HD], w["qn"]), pos), qg[..., HD:]
    k = _rope64(_norm64((x @ _wide4(*w["k"])[0].T).reshape(s, KH, HD), w["kn"]), pos)
    v = (x @ _wide4(*w["v"])[0].T).reshape(s, KH, HD)
    mask = torch.arange(pos + s, device="cuda")[None] > torch.arange(pos, pos + s, device="cuda")[:, None]
    ctx = torch.empty((s, H, HD), dtype=F64, device="cuda")
    for h in range(H):
        g = h // (H // KH)
        kk, vv = torch.cat((kc[g].to(F64), k[:, g])), torch.cat((vc[g].to(F64), v[:, g]))
        sc = (q[:, h] @ kk.T) / math.sqrt(HD)
        ctx[:, h] = torch.softmax(sc.masked_fill(mask, -math.inf), 1) @ vv
    return (ctx * torch.sigmoid(gate)).reshape(s, H * HD) @ _wide4(*w["o"])[0].T


def _gdn64(x, w, params):
    """Rows x of a new sequence."""
    s = x.shape[0]
    qkv, z = x @ _wide4(*w["qkv"])[0].T, (x @ _wide4(*w["z"])[0].T).reshape(s, GVH, GVD)
    past = torch.cat((torch.zeros((GCK - 1, GCD), dtype=F64, device="cuda"), qkv))
    c = sum(past[j:j + s] * w["conv"][:, j].to(F64) for j in range(GCK))
    c = torch.nn.functional.silu(c)
    kd = GKH * GKD
    q, k, v = c[:, :kd].reshape(s, GKH, GKD), c[:, kd:2 * kd].reshape(s, GKH, GKD), c[:, 2 * kd:].reshape(s, GVH, GVD)
    q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + EPS) / math.sqrt(GKD)
    k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + EPS)
    q, k = (t.repeat_interleave(GVH // GKH, 1) for t in (q, k))
    decay, beta = params[:, :GVH].to(F64), params[:, GVH:2 * GVH].to(F64)
    S = torch.zeros((GVH, GKD, GVD), dtype=F64, device="cuda")
    y = torch.empty((s, GVH, GVD), dtype=F64, device="cuda")
    for t in range(s):
        S = S * decay[t][:, None, None]
        d = (v[t] - (S * k[t][:, :, None]).sum(1)) * beta[t][:, None]
        S = S + k[t][:, :, None] * d[:, None, :]
        y[t] = (S * q[t][:, :, None]).sum(1)
    y = y * torch.rsqrt((y * y).mean(-1, keepdim=True) + EPS) * w["gnorm"].to(F64) * torch.nn.functional.silu(z)
    return y.reshape(s, GVH * GVD) @ _wide4(*w["out"])[0].T


def exact(case, seed):
    p = case["path"]
    if p == "gemv":
        return _acts(case["S"], case["I"], seed, 2).to(F64) @ _wide4(*_int4(1, case["O"], case["I"], seed, 1))[0].T
    if p == "topk":
        y = _acts(1, case["I"], seed, 2)[0].to(F64) @ _wide4(*_int4(1, case["O"], case["I"], seed, 1))[0].T
        val, idx = y.topk(case["k"])
        return y, val, idx.to(torch.int32)
    if p in ("moe", "prefill"):
        ex, s = _experts(case["E"], case["D"], case["I"], seed, 10), case.get("S", 1)
        router = _router(case["E"], case["D"], case["router"], seed, 3)[1]()
        out, v, ids, sh = _moe64(_acts(s, case["D"], seed, 2).to(F64), router, ex, case["K"])
        return out, torch.cat((v[0], sh)) if p == "moe" else v, ids.to(torch.int32) if p == "prefill" else ids[0].to(torch.int32)
    if p == "experts":
        ex, x = _experts(E, D, I, seed, 10), _acts(case["S"], D, seed, 2).to(F64)
        ys = [_mlp(x[torch.from_numpy(tok).cuda()], ex, e)
              for ch in _chunks(_route_ids(case["S"], seed, 4)) for e, tok in ch]
        return torch.cat(ys + [_mlp(x, ex, E)])
    if p == "gqa":
        w = _gqa_weights(seed, 20)
        return _gqa64(_acts(case["S"], D, seed, 2).to(F64), w, *_cache(seed, 40, case["pos"])).reshape(-1)
    if p == "gdn":
        w, x = _gdn_weights(seed, 20), _acts(case["S"], D, seed, 2)
        return _gdn64(x.to(F64), w, _gdn_params(w, x)).reshape(-1)
    x = _normal(D, 1.0, seed, 2).to(F64)[None]
    for n in range(4):
        tag = 100 * (n + 1)
        nx = _norm64(x, _normal(D, 0.1, seed, tag + 61))
        if n == 3:
            x = x + _gqa64(nx, _gqa_weights(seed, tag), *_cache(seed, 40, case["pos"]))
        else:
            w = _gdn_weights(seed, tag)
            a = nx @ _wide8(*w["a"]).T + w["dtb"].to(F64)
            decay = torch.exp(-torch.exp(w["alog"].to(F64)) * torch.nn.functional.softplus(a))
            x = x + _gdn64(nx, w, torch.cat((decay, torch.sigmoid(nx @ _wide8(*w["b"]).T)), 1))
        router = _router(E, D, "int8", seed, tag + 60)[1]()
        x = x + _moe64(_norm64(x, _normal(D, 0.1, seed, tag + 62)), router, _experts(E, D, I, seed, tag + 50), K)[0]
    return x[0]
