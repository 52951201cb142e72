"""The work whose time matters to a user of the library, each case through public entry points.

The shapes are DeepSeek-OCR's decoder (hidden 1280, 64 routed experts 1792x1280 + 1280x896, top 6 and 2
shared experts, 10 heads x 128, dense layer 1280 x 6848, head 129280 x 1280) and, among the drawn cases, the
smaller shapes of the test suite. Weights are N(0, 0.02) and hidden states N(0, 1), as in bench.py.

Kinds:
  expert   ds_expert_forward_fused_int4: one expert of the per-function drop-in path, host in and out
  linear   ds_linear_nobias_bf16 with many rows: the drop-in path's prefill projections, host in and out
  layer    ds_hip_layer_forward: one MoE layer for one token, in device memory
  attn     ds_hip_attn_forward: the attention half of a decoder layer for one token
  dense    ds_hip_dense_forward: the decoder's first MLP for one token
  stack    ds_hip_stack_run: MoE layers and the argmax head, several steps on their own inputs
  decoder  ds_hip_stack_run: whole decoder steps, each fed with the token before it
  prefill  ds_hip_layer_prefill: one MoE layer for a prompt's tokens
"""
import ctypes as C
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_DEV = "cuda"
_THREADS = 16  # the reference's own limit, which its decode always uses


def _product():
    name = "ds_ocr_amd"
    if name not in sys.modules:
        root = os.getcwd()
        spec = importlib.util.spec_from_file_location(name, os.path.join(root, "ds-ocr_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


_SHAPE = {"hidden": 1280, "inter": 896, "experts": 64, "top_k": 6, "shared": 2}
_SMALL = {"hidden": 256, "inter": 128, "experts": 16, "top_k": 6, "shared": 2}
_MID = {"hidden": 512, "inter": 256, "experts": 32, "top_k": 6, "shared": 2}
_HEADS = {"heads": 10, "head_dim": 128, "qk_norm": False}


def listed():
    return [
        # a drop-in caller's routed expert: 66 such calls per token
        {"name": "expert_host", "kind": "expert", "hidden": 1280, "inter": 896},
        # a drop-in caller's prefill projection of one page (662 tokens)
        {"name": "linear_host_662", "kind": "linear", "rows": 662, "hidden": 1280, "out": 1280},
        # a caller that owns the decoder loop: one MoE layer at a time
        {"name": "layer_cfg", "kind": "layer", **_SHAPE, "route": 1, "sim": False, "residual": True},
        # the same with the reference's bf16 simulation and its decode router
        {"name": "layer_sim_decode", "kind": "layer", **_SHAPE, "route": 0, "sim": True, "residual": True},
        # attention early in the answer to one page, and late in a long document
        {"name": "attn_701", "kind": "attn", "hidden": 1280, **_HEADS, "pos": 701, "max_seq": 2048, "prefill": 0,
         "window": 0},
        {"name": "attn_7001", "kind": "attn", "hidden": 1280, **_HEADS, "pos": 7001, "max_seq": 7680, "prefill": 0,
         "window": 0},
        # the decoder's layer 0
        {"name": "dense_6848", "kind": "dense", "hidden": 1280, "inter": 6848, "residual": True},
        # the batch-1 decode hot path
        {"name": "stack_11x8", "kind": "stack", **_SHAPE, "layers": 11, "vocab": 129280, "route": 1, "steps": 8},
        # whole decoder steps after a page of 1000 positions, as the decode loop runs them
        {"name": "decoder_12x8", "kind": "decoder", **_SHAPE, **_HEADS, "layers": 11, "dense": 6848, "vocab": 129280,
         "route": 0, "pos": 1000, "steps": 8},
        # a thumbnail's prompt, one page, and a batch of tiles
        {"name": "prefill_77", "kind": "prefill", **_SHAPE, "tokens": 77, "route": 0, "residual": True},
        {"name": "prefill_662", "kind": "prefill", **_SHAPE, "tokens": 662, "route": 1, "residual": True},
        {"name": "prefill_3001", "kind": "prefill", **_SHAPE, "tokens": 3001, "route": 0, "residual": True},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["expert", "linear", "layer", "attn", "attn", "dense", "stack", "decoder", "prefill", "prefill"])
    shape = dict(rng.choice([_SHAPE, _SHAPE, _SMALL, _MID]))
    if kind == "expert":
        return {"kind": kind, "hidden": _log(rng, 64, 2048), "inter": _log(rng, 32, 1792)}
    if kind == "linear":
        return {"kind": kind, "rows": _log(rng, 2, 1500), "hidden": _log(rng, 64, 2048), "out": _log(rng, 64, 4000)}
    if kind == "layer":
        return {"kind": kind, **shape, "route": rng.randrange(2), "sim": rng.random() < 0.3,
                "residual": rng.random() < 0.7}
    if kind == "attn":
        max_seq = _log(rng, 64, 7680)
        pos = _log(rng, 1, max_seq) - 1
        windowed = rng.random() < 0.3
        return {"kind": kind, **rng.choice([{"hidden": 1280, **_HEADS}, {"hidden": 1280, **_HEADS},
                                            {"hidden": 256, "heads": 2, "head_dim": 128, "qk_norm": True},
                                            {"hidden": 512, "heads": 8, "head_dim": 64, "qk_norm": False}]),
                "pos": pos, "max_seq": max_seq, "prefill": pos // 2 if windowed else 0,
                "window": _log(rng, 1, 1024) if windowed else 0}
    if kind == "dense":
        return {"kind": kind, "hidden": 128 * rng.randrange(1, 17), "inter": 8 * _log(rng, 16, 1024),
                "residual": rng.random() < 0.5}
    if kind == "stack":
        return {"kind": kind, **shape, "layers": rng.randrange(1, 9), "vocab": _log(rng, 2000, 129280),
                "route": rng.randrange(2), "steps": rng.randrange(1, 9)}
    if kind == "decoder":
        heads = {1280: 10, 512: 4, 256: 2}[shape["hidden"]]
        return {"kind": kind, **shape, "heads": heads, "head_dim": 128, "qk_norm": rng.random() < 0.3,
                "layers": rng.randrange(1, 5), "dense": 8 * _log(rng, 16, 856), "vocab": _log(rng, 2000, 129280),
                "route": rng.randrange(2), "pos": _log(rng, 1, 3000), "steps": rng.randrange(1, 7)}
    return {"kind": kind, **shape, "tokens": _log(rng, 1, 3001), "route": rng.randrange(2),
            "residual": rng.random() < 0.5}


# ------------------------------------------------------------------ what a program has in hand

class _Handle:
    """A library handle (and what it borrows), destroyed with the object."""

    def __init__(self, ptr, destroy, borrows=()):
        if not ptr:
            raise RuntimeError(_product().load().ds_hip_last_error().decode())
        self.ptr, self._destroy, self._borrows = ptr, destroy, borrows

    def __del__(self):
        self._destroy(self.ptr)


class _Memory:
    """Device memory of a handle as an array that torch can read; keeps the handle."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2}


class _Blocks:
    """Host INT8 blocks of the library, freed with the object."""

    def __init__(self, blocks):
        self.blocks = blocks

    def __del__(self):
        for b in self.blocks:
            _product().load().ds_int4_block_free(C.byref(b))


class _State:
    pass


def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(seed)


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=_DEV) * std


def _weight(g, *shape):
    return _normal(g, *shape, std=0.02).to(torch.bfloat16)


def _bits(t):
    """A bf16 tensor's bits as a host array, the form the library takes host weights in."""
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


def _layer_weights(g, c):
    H, I, E, SI = c["hidden"], c["inter"], c["experts"], c["shared"] * c["inter"]
    rf = _normal(g, E, H, std=0.02)
    return {"rf": rf, "rb": rf.to(torch.bfloat16), "gu": _weight(g, E, 2 * I, H), "dn": _weight(g, E, H, I),
            "sgu": _weight(g, 2 * SI, H), "sdn": _weight(g, H, SI)}


def _attn_weights(g, c):
    H, qd = c["hidden"], c["heads"] * c["head_dim"]
    w = {k: _weight(g, qd, H) for k in ("wq", "wk", "wv")}
    w["wo"] = _weight(g, H, qd)
    w["n1"], w["n2"] = (1 + _normal(g, H, std=0.1) for _ in range(2))
    w["qn"], w["kn"] = (1 + _normal(g, c["head_dim"], std=0.1) for _ in range(2)) if c["qk_norm"] else (None, None)
    return w


def _dense_weights(g, H, I):
    return _weight(g, I, H), _weight(g, I, H), _weight(g, H, I)


def _kv(g, c, rows):
    qd = c["heads"] * c["head_dim"]
    return _normal(g, rows, qd), _normal(g, rows, qd)


def _make_layer(P, c, w):
    L = P.load()
    H, I, E = c["hidden"], c["inter"], c["experts"]
    h = _Handle(L.ds_hip_layer_create(H, I, E, c["top_k"], c["shared"] * I), L.ds_hip_layer_destroy)
    torch.cuda.synchronize()
    P.check(L.ds_hip_layer_set_router_dev(h.ptr, w["rf"].data_ptr(), w["rb"].data_ptr()), "router")
    for e in range(E):
        P.check(L.ds_hip_layer_quantize_expert(h.ptr, e, w["gu"][e].data_ptr(), w["dn"][e].data_ptr()), "expert")
    P.check(L.ds_hip_layer_quantize_expert(h.ptr, -1, w["sgu"].data_ptr(), w["sdn"].data_ptr()), "shared")
    P.check(L.ds_hip_sync(), "sync")
    return h


_ROPE, _EPS = 10000.0, 1e-6


def _make_attn(P, c, w, max_seq, prefill, window, cached):
    """The handle and its K and V caches as tensors, the first rows holding the cached positions."""
    L = P.load()
    host = [_bits(w[k]) for k in ("wq", "wk", "wv", "wo")]
    host += [w[k].cpu().numpy() if w[k] is not None else None for k in ("n1", "n2", "qn", "kn")]
    h = _Handle(L.ds_hip_attn_create(c["hidden"], c["heads"], c["head_dim"], max_seq, _EPS, _ROPE,
                                     *[a.ctypes.data if a is not None else None for a in host]), L.ds_hip_attn_destroy)
    P.check(L.ds_hip_attn_set_window(h.ptr, prefill, window), "window")
    k, v, stride = C.c_void_p(), C.c_void_p(), C.c_int()
    P.check(L.ds_hip_attn_kv(h.ptr, C.byref(k), C.byref(v), C.byref(stride)), "caches")
    P.check(L.ds_hip_sync(), "sync")
    caches = [torch.as_tensor(_Memory(h, p.value, (max_seq, stride.value)), device=_DEV) for p in (k, v)]
    for t, rows in zip(caches, cached):
        t[:rows.shape[0], :rows.shape[1]] = rows
    return h, caches


def _make_dense(P, H, I, w):
    L = P.load()
    host = [_bits(t) for t in w]
    return _Handle(L.ds_hip_dense_create(H, I, *[a.ctypes.data for a in host]), L.ds_hip_dense_destroy)


def prepare(case, seed):
    P = _product()
    L = P.load()
    P.check(L.ds_hip_init(), "init")
    L.ds_set_threads(_THREADS)
    c, g, s = case, _gen(seed), _State()
    s.P, s.L, s.c = P, L, case
    H = c["hidden"]
    if c["kind"] == "expert":
        gu, dn = _weight(g, 2 * c["inter"], H), _weight(g, H, c["inter"])
        s.x, s.out = _normal(g, H).cpu().numpy(), np.empty(H, np.float32)
        s.gu, s.dn = P.Int4Block(), P.Int4Block()
        for b, w in ((s.gu, gu), (s.dn, dn)):
            if L.ds_int4_quantize_bf16(C.byref(b), _bits(w), *w.shape):
                raise RuntimeError(L.ds_hip_last_error().decode())
        s.keep = _Blocks([s.gu, s.dn])
    elif c["kind"] == "linear":
        s.w = _bits(_weight(g, c["out"], H))
        s.x, s.out = _normal(g, c["rows"], H).cpu().numpy(), np.empty((c["rows"], c["out"]), np.float32)
        P.check(L.ds_hip_register_weights(s.w.ctypes.data, s.w.nbytes), "register")
        s.keep = _Registered(L, s.w)
    elif c["kind"] in ("layer", "prefill"):
        T = c.get("tokens", 1)
        s.layer = _make_layer(P, c, _layer_weights(g, c))
        s.x, s.out = _normal(g, T, H), torch.empty(T, H, device=_DEV)
        s.idx = torch.empty(T, c["top_k"], dtype=torch.int32, device=_DEV)
        s.w = torch.empty(T, c["top_k"], device=_DEV)
    elif c["kind"] == "attn":
        w = _attn_weights(g, c)
        s.attn, s.caches = _make_attn(P, c, w, c["max_seq"], c["prefill"], c["window"], _kv(g, c, c["pos"]))
        s.x, s.h, s.n = _normal(g, H), torch.empty(H, device=_DEV), torch.empty(H, device=_DEV)
    elif c["kind"] == "dense":
        s.dense = _make_dense(P, H, c["inter"], _dense_weights(g, H, c["inter"]))
        s.x, s.out = _normal(g, H), torch.empty(H, device=_DEV)
    else:
        layers = [_make_layer(P, c, _layer_weights(g, c)) for _ in range(c["layers"])]
        head = _weight(g, c["vocab"], H)
        s.tokens = torch.empty(c["steps"], dtype=torch.int32, device=_DEV)
        s.hidden = np.empty(H, np.float32)
        s.x = _normal(g, c["steps"] if c["kind"] == "stack" else 1, H)
        torch.cuda.synchronize()
        arr = (C.c_void_p * len(layers))(*[h.ptr for h in layers])
        borrows = [layers, head, s.x, s.tokens]
        s.stack = _Handle(L.ds_hip_stack_create(arr, len(layers), head.data_ptr(), c["vocab"], c["route"]),
                          L.ds_hip_stack_destroy, borrows)
        stride = H
        if c["kind"] == "decoder":
            dense = _make_dense(P, H, c["dense"], _dense_weights(g, H, c["dense"]))
            embed = _weight(g, c["vocab"], H)
            made = [_make_attn(P, c, _attn_weights(g, c), c["pos"] + c["steps"], 0, 0, _kv(g, c, c["pos"]))
                    for _ in range(c["layers"] + 1)]
            norm = (1 + _normal(g, H, std=0.1)).cpu().numpy()
            s.caches = [t for _, caches in made for t in caches]
            borrows += [dense, embed, [h for h, _ in made]]
            stride = 0
            P.check(L.ds_hip_stack_set_dense(s.stack.ptr, dense.ptr), "dense")
            at = (C.c_void_p * len(made))(*[h.ptr for h, _ in made])
            P.check(L.ds_hip_stack_set_attention(s.stack.ptr, at, len(made), norm.ctypes.data, _EPS, c["pos"], 0), "attn")
            P.check(L.ds_hip_stack_set_embedding(s.stack.ptr, embed.data_ptr(), c["vocab"]), "embedding")
        torch.cuda.synchronize()
        P.check(L.ds_hip_stack_bind(s.stack.ptr, s.x.data_ptr(), stride, s.x.shape[0], s.tokens.data_ptr(), c["steps"]),
                "bind")
    torch.cuda.synchronize()
    P.check(L.ds_hip_sync(), "sync")
    return s


class _Registered:
    """A registered host weight array: its device copy is dropped with the object."""

    def __init__(self, L, w):
        self.L, self.w = L, w

    def __del__(self):
        self.L.ds_hip_weights_changed(self.w.ctypes.data)


def run(state):
    s, c, L, check = state, state.c, state.L, state.P.check
    kind = c["kind"]
    if kind == "expert":
        L.ds_expert_forward_fused_int4(s.out, s.x, C.byref(s.gu), C.byref(s.dn), c["hidden"], c["inter"], None, None,
                                       None, None)
        return s.out
    if kind == "linear":
        L.ds_linear_nobias_bf16(s.out.reshape(-1), s.x.reshape(-1), s.w.reshape(-1), c["rows"], c["hidden"], c["out"])
        return s.out
    if kind == "layer":
        if c["sim"]:
            s.P.set_bf16sim(True)
        try:
            check(L.ds_hip_layer_forward(s.layer.ptr, s.out.data_ptr(), s.x.data_ptr(), c["route"], int(c["residual"]),
                                         s.idx.data_ptr(), s.w.data_ptr()), "layer")
        finally:
            if c["sim"]:
                s.P.set_bf16sim(False)
        return {"out": s.out, "idx": s.idx, "w": s.w}
    if kind == "prefill":
        check(L.ds_hip_layer_prefill(s.layer.ptr, s.out.data_ptr(), s.x.data_ptr(), c["tokens"], c["route"],
                                     int(c["residual"]), s.idx.data_ptr(), s.w.data_ptr()), "prefill")
        return {"out": s.out, "idx": s.idx, "w": s.w}
    if kind == "attn":
        check(L.ds_hip_attn_forward(s.attn.ptr, s.h.data_ptr(), s.n.data_ptr(), s.x.data_ptr(), c["pos"]), "attention")
        return {"h": s.h, "n": s.n, "k": s.caches[0], "v": s.caches[1]}
    if kind == "dense":
        check(L.ds_hip_dense_forward(s.dense.ptr, s.out.data_ptr(), s.x.data_ptr(), int(c["residual"])), "dense")
        return s.out
    check(L.ds_hip_stack_reset(s.stack.ptr), "reset")
    check(L.ds_hip_stack_run(s.stack.ptr, c["steps"]), "steps")
    check(L.ds_hip_stack_hidden(s.stack.ptr, s.hidden), "hidden")
    got = {"tokens": s.tokens, "hidden": s.hidden}
    if kind == "decoder":
        got["kv"] = s.caches
    return got


# ------------------------------------------------------------------ what a pass cannot do without

def _layer_work(c, T):
    H, I, E, K, SI = c["hidden"], c["inter"], c["experts"], c["top_k"], c["shared"] * c["inter"]
    hit = E * (1 - (1 - K / E) ** T)  # experts that T tokens' choices reach
    expert = 3 * H * I + 8 * (2 * I + H)
    shared = 3 * H * SI + 8 * (2 * SI + H)
    router = E * H * (4 if c["route"] else 2)
    flops = 2.0 * T * (3 * H * (K * I + SI) + E * H)
    return hit * expert + shared + router, flops


def _attn_work(c, pos, prefill, window):
    H, qd = c["hidden"], c["heads"] * c["head_dim"]
    n = pos + 1
    if window and pos >= prefill:
        n = min(n, prefill + min(window, n - prefill))
    return 2.0 * 4 * H * qd + 8.0 * H + 2.0 * 4 * n * qd, 2.0 * 4 * H * qd + 4.0 * n * qd


def work(case):
    c = case
    H, kind = c["hidden"], c["kind"]
    if kind == "expert":
        I = c["inter"]
        return {"bytes": 3.0 * H * I + 8 * (2 * I + H) + 8 * H, "flops": 6.0 * H * I}
    if kind == "linear":
        return {"bytes": 2.0 * H * c["out"] + 4.0 * c["rows"] * (H + c["out"]), "flops": 2.0 * H * c["out"] * c["rows"]}
    if kind in ("layer", "prefill"):
        T = c.get("tokens", 1)
        b, f = _layer_work(c, T)
        return {"bytes": b + 8.0 * T * (H + c["top_k"]), "flops": f}
    if kind == "attn":
        b, f = _attn_work(c, c["pos"], c["prefill"], c["window"])
        return {"bytes": b + 12.0 * H, "flops": f}
    if kind == "dense":
        return {"bytes": 6.0 * H * c["inter"] + 8.0 * H, "flops": 6.0 * H * c["inter"]}
    b, f = _layer_work(c, 1)
    b, f = b * c["layers"], f * c["layers"]
    # the head: its argmax is exact, and half of its bf16 bytes suffice to bound all but a few rows
    b, f = b + 1.0 * c["vocab"] * H, f + 2.0 * c["vocab"] * H
    if kind == "decoder":
        a = [_attn_work(c, c["pos"] + i, 0, 0) for i in range(c["steps"])]
        n = c["layers"] + 1
        b += 6.0 * H * c["dense"] + n * sum(x for x, _ in a) / len(a)
        f += 6.0 * H * c["dense"] + n * sum(x for _, x in a) / len(a)
    return {"bytes": b * c["steps"], "flops": f * c["steps"]}


def tolerance(case):
    """About four times what the start shows against exact()."""
    kind = case["kind"]
    if kind == "expert" or (kind == "layer" and case["sim"]):
        return "exact"  # the reference's own order, bit for bit
    if kind == "prefill":
        return {"rel": 2e-4, "max": 2e-3}  # activations on a 16-bit grid
    if kind == "stack":
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "decoder":
        return {"rel": 4e-5, "max": 4e-4}
    return {"rel": 2e-6, "max": 2e-5}  # 32-bit sums


# ------------------------------------------------------------------ the same in 64 bits

def _fast_exp(x):
    """The Schraudolph exponential that the model is defined with: linear between powers of two."""
    i = torch.clamp((12102203.0 * x + 1064866805.0) / 8388608.0, min=0.0)
    e = torch.floor(i)
    v = torch.exp2(e - 127.0) * (1.0 + (i - e))
    return torch.where(x < -88.0, torch.zeros_like(v), torch.where(x > 88.0, torch.full_like(v, 1e38), v))


def _round16(x, on):
    if not on:
        return x
    return ((x.float().contiguous().view(torch.int32) + 0x8000) & -65536).view(torch.float32).double()


def _quantized(w):
    """The values that 8-bit codes with a scale and an offset per row stand for."""
    w = w.float()
    lo, hi = w.amin(-1, keepdim=True), w.amax(-1, keepdim=True)
    # 255 as a tensor: torch turns a division by a number into a product with its reciprocal
    scale = torch.clamp((hi - lo) / torch.full_like(lo, 255.0), min=1e-10)
    u = torch.clamp(torch.floor((w - lo) * (torch.ones_like(scale) / scale) + 0.5), 0, 255)
    return scale.double() * u.double() + lo.double()


def _swiglu(g, u):
    return g / (1.0 + _fast_exp(-g)) * u


def _expert64(x, gu, dn, sim=False):
    """x [n, H]; gu, dn: bf16 weights of one expert."""
    y = _round16(x @ _quantized(gu).T, sim)
    g, u = y.chunk(2, -1)
    return _round16(_round16(_swiglu(g, u), sim) @ _quantized(dn).T, sim)


def _route64(x, w, c):
    """Expert indices in rank order and their weights for x [T, H]."""
    if c["route"]:
        v, idx = torch.topk(x @ w["rf"].double().T, c["top_k"])
        return idx, torch.softmax(v, -1)
    s = x @ w["rb"].double().T
    e = _fast_exp(s - s.amax(-1, keepdim=True))
    v, idx = torch.topk(e / e.sum(-1, keepdim=True), c["top_k"])
    return idx, v


def _moe64(x, w, c, sim=False):
    idx, p = _route64(x, w, c)
    out = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        t, k = torch.nonzero(idx == e, as_tuple=True)
        out.index_add_(0, t, p[t, k, None] * _expert64(x[t], w["gu"][e], w["dn"][e], sim))
    out += _expert64(x, w["sgu"], w["sdn"], sim)
    return out, idx.int(), p


def _norm64(x, w):
    return x * w.double() / torch.sqrt((x * x).mean(-1, keepdim=True) + _EPS)


def _attn64(x, w, c, kc, vc, pos, prefill, window):
    """One token; writes its rows into kc and vc ([max_seq, qd], f64) and returns h and its norm."""
    nh, hd = c["heads"], c["head_dim"]
    xn = _norm64(x, w["n1"])
    q, k, v = (w[n].double() @ xn for n in ("wq", "wk", "wv"))
    q, k = q.view(nh, hd), k.view(nh, hd)
    if c["qk_norm"]:
        q, k = _norm64(q, w["qn"]), _norm64(k, w["kn"])
    half = hd // 2
    # the angles are part of the model: 32-bit frequencies times 32-bit positions
    freq = np.float32(1) / np.power(np.float32(_ROPE), np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd))
    a = torch.from_numpy((np.float32(pos) * freq).astype(np.float64)).to(x.device)
    cs, sn = torch.cos(a), torch.sin(a)
    q, k = (torch.cat([t[:, :half] * cs - t[:, half:] * sn, t[:, :half] * sn + t[:, half:] * cs], -1) for t in (q, k))
    kc[pos, :nh * hd], vc[pos, :nh * hd] = k.reshape(-1), v
    at = torch.arange(pos + 1, device=x.device)
    if window and pos >= prefill:
        at = at[(at < prefill) | (at > pos - window)]
    K, V = (t[at, :nh * hd].view(-1, nh, hd) for t in (kc, vc))
    s = torch.einsum("hd,nhd->hn", q, K) / math.sqrt(hd)
    # a running softmax with that exponential, which does not turn sums into products: in order
    before = torch.cummax(torch.cat([torch.full_like(s[:, :1], -1e30), s], -1), -1).values[:, :-1]
    new = s > before
    f = _fast_exp(torch.where(new, before - s, s - before))
    fall = torch.where(new, f, torch.ones_like(f))
    later = torch.cat([torch.flip(torch.cumprod(torch.flip(fall, [-1]), -1), [-1])[:, 1:], torch.ones_like(s[:, :1])], -1)
    coef = torch.where(new, torch.ones_like(f), f) * later
    o = torch.einsum("hn,nhd->hd", coef, V) / coef.sum(-1, keepdim=True)
    h = x + w["wo"].double() @ o.reshape(-1)
    return h, _norm64(h, w["n2"])


def exact(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    H = c["hidden"]
    if kind == "expert":
        gu, dn = _weight(g, 2 * c["inter"], H), _weight(g, H, c["inter"])
        return _expert64(_normal(g, H)[None].double(), gu, dn)[0].cpu().numpy()
    if kind == "linear":
        w = _weight(g, c["out"], H).double()
        return (_normal(g, c["rows"], H).double() @ w.T).cpu().numpy()
    if kind in ("layer", "prefill"):
        w = _layer_weights(g, c)
        x = _normal(g, c.get("tokens", 1), H).double()
        out, idx, p = _moe64(x, w, c, c.get("sim", False))
        return {"out": x + out if c["residual"] else out, "idx": idx, "w": p}
    if kind == "attn":
        w = _attn_weights(g, c)
        caches = []
        for rows in _kv(g, c, c["pos"]):
            t = torch.zeros(c["max_seq"], rows.shape[1], dtype=torch.float64, device=_DEV)
            t[:c["pos"]] = rows
            caches.append(t)
        h, n = _attn64(_normal(g, H).double(), w, c, *caches, c["pos"], c["prefill"], c["window"])
        return {"h": h, "n": n, "k": caches[0], "v": caches[1]}
    if kind == "dense":
        wg, wu, wd = (t.double() for t in _dense_weights(g, H, c["inter"]))
        x = _normal(g, H).double()
        y = wd @ _swiglu(wg @ x, wu @ x)
        return x + y if c["residual"] else y
    layers = [_layer_weights(g, c) for _ in range(c["layers"])]
    head = _weight(g, c["vocab"], H)
    x = _normal(g, c["steps"] if kind == "stack" else 1, H).double()
    if kind == "stack":
        for w in layers:
            x = x + _moe64(x, w, c)[0]
        return {"tokens": (x @ head.double().T).argmax(-1).int(), "hidden": x[-1].cpu().numpy()}
    wg, wu, wd = (t.double() for t in _dense_weights(g, H, c["dense"]))
    embed = _weight(g, c["vocab"], H)
    attn, caches = [], []
    for _ in range(c["layers"] + 1):
        attn.append(_attn_weights(g, c))
        caches.append([torch.cat([t.double(), torch.zeros(c["steps"], t.shape[1], dtype=torch.float64, device=_DEV)])
                       for t in _kv(g, c, c["pos"])])
    norm = (1 + _normal(g, H, std=0.1))
    x, tokens, head64 = x[0], [], head.double()
    for i in range(c["steps"]):
        h, n = _attn64(x, attn[0], c, *caches[0], c["pos"] + i, 0, 0)
        x = h + wd @ _swiglu(wg @ n, wu @ n)
        for w, a, kv in zip(layers, attn[1:], caches[1:]):
            h, n = _attn64(x, a, c, *kv, c["pos"] + i, 0, 0)
            x = h + _moe64(n[None], w, c)[0][0]
        hidden = x
        tokens.append(int((head64 @ _norm64(x, norm)).argmax()))
        x = embed[tokens[-1]].double()
    return {"tokens": torch.tensor(tokens, dtype=torch.int32), "hidden": hidden.cpu().numpy(),
            "kv": [t for kv in caches for t in kv]}
