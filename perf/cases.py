"""The work this framework is used for, as cases to time and to compare.

A decode step is what a user runs: the whole token step through the
backend's ops table and through the graph and batched decoders, and its parts
one at a time through the device library's entry points: the matvecs of a
layer in each weight format (batch 1 and several vectors), the output head
and the embedding gather, the attention over the f16 cache, and the CPU hot
table's matvec. Sizes are those of bench.py (the 7B and 70B Llama shapes and
the hot table's) and of tests/ (the two-layer model, the random matvec and
attention shapes).

Weights are random GGUF blocks with the value ranges of host/vbs_synth.c,
made on the GPU from the case's seed; x and q are N(0,1) and the caches f16
N(0,1).
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "verum-bespoke-singularity_amd"))
import vbs_gfx950 as V  # noqa: E402

DEV = "cuda"
TYPES = {"Q4_0": V.Q4_0, "Q4_1": V.Q4_1, "Q8_0": V.Q8_0, "Q4_K": V.Q4_K, "Q6_K": V.Q6_K,
         "F16": V.F16, "F32": V.F32, "LNS8": V.LNS8}
# hidden, ffn, query heads, kv heads, head size, vocabulary
GEO = {"7b": (4096, 11008, 32, 8, 128, 32000), "70b": (8192, 28672, 64, 8, 128, 32000),
       "small": (256, 512, 4, 2, 64, 512)}
EPS, THETA = 1e-5, 10000.0
ROLES = ("q", "k", "v", "o", "gate", "up", "down")


def listed():
    return [
        # the smallest whole step, through the ops table: the two-layer model of the tests,
        # where launches, host work and latency are all there is
        {"name": "ops_step_small", "kind": "ops", "layers": 2, "hidden": 256, "ffn": 512,
         "heads": 4, "kv_heads": 2, "hd": 64, "vocab": 512, "mix": "Q4_K_M", "pos": 40},
        # one token of a 7B Q4_K_M model at a context of 2048, logits returned
        {"name": "decode_7b", "kind": "decode", "geo": "7b", "layers": 32, "pos": 2048},
        # one step of eight sequences of the 70B shape at a context of 8192 (four of its layers)
        {"name": "batch8_70b", "kind": "bdecode", "geo": "70b", "layers": 4, "pos": 8191, "batch": 8},
        # the seven matvecs of a 7B layer, one graph launch, as bench.py issues them
        {"name": "layer_q4_k_7b", "kind": "layer", "type": "Q4_K", "hidden": 4096, "kv": 4096, "ffn": 11008},
        # the same in the format of a less compressed model file
        {"name": "layer_q8_0_7b", "kind": "layer", "type": "Q8_0", "hidden": 4096, "kv": 4096, "ffn": 11008},
        # an unquantised matrix of a mixed-type model
        {"name": "linear_f16", "kind": "linear", "type": "F16", "rows": 11008, "cols": 4096, "acc": False},
        # an odd matrix: rows of 177 blocks of 32 (no multiple of 256), added to y
        {"name": "linear_q4_0_ragged", "kind": "linear", "type": "Q4_0", "rows": 2049, "cols": 5664, "acc": True},
        # the 70B layer matvec set for eight sequences, grouped as the batched decoder groups it
        {"name": "batch8_layer_70b", "kind": "blayer", "type": "Q4_K_M", "hidden": 8192, "kv": 1024, "ffn": 28672,
         "batch": 8},
        # several sequences over a model in Q8_0
        {"name": "batch8_layer_q8_0_7b", "kind": "blayer", "type": "Q8_0", "hidden": 4096, "kv": 1024, "ffn": 11008,
         "batch": 8},
        # the output head, and the gather of 64 token embeddings
        {"name": "head_gather_q6_k", "kind": "head", "type": "Q6_K", "vocab": 32000, "dim": 4096, "ids": 64},
        # attention with heads of 64 over a ragged context
        {"name": "attention_hd64", "kind": "attention", "heads": 32, "kv_heads": 8, "hd": 64, "seq": 3001, "layer": 1},
        # the CPU hot table's Q8_0 matvec on resident buffers, with its activations quantised
        {"name": "hot_q8_0", "kind": "hot", "type": "Q8_0", "rows": 4096, "cols": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cols(rng, t, lo=32, hi=28672):
    """A row length of type t: mostly whole super-blocks, as models have them, and odd counts of
    32-element blocks (any count for the types without blocks)."""
    if t in ("F16", "F32") and rng.random() < 0.3:
        return max(1, _log(rng, lo, hi))
    e = 256 if t in ("Q4_K", "Q6_K") or rng.random() < 0.4 else 32
    return e * max(1, _log(rng, lo, hi) // e)


def draw(rng):
    kind = rng.choice(["ops", "decode", "bdecode", "layer", "linear", "linear", "blayer", "batch",
                       "head", "attention", "hot"])
    c = {"kind": kind}
    if kind == "ops":
        hd, kvh = rng.choice([32, 64, 128]), rng.choice([1, 2, 4])
        heads = kvh * rng.choice([1, 2, 4])
        c.update(layers=rng.randint(1, 4), hidden=256 * rng.randint(1, 4), ffn=256 * rng.randint(1, 8),
                 heads=heads if heads * hd % 256 == 0 else heads * (256 // math.gcd(256, heads * hd)),
                 kv_heads=kvh, hd=hd, vocab=16 * rng.randint(16, 128),
                 mix=rng.choice(["Q4_K_M", "Q8_0", "Q4_0"]), pos=_log(rng, 1, 500))
    elif kind == "decode":
        g = rng.choice(["small", "7b", "70b"])
        c.update(geo=g, layers=rng.randint(1, 4), pos=_log(rng, 1, 8000))
    elif kind == "bdecode":
        c.update(geo=rng.choice(["7b", "70b"]), layers=rng.randint(1, 3), pos=_log(rng, 8, 8000),
                 batch=rng.randint(1, 8))
    elif kind in ("layer", "blayer"):
        types = ["Q4_0", "Q4_1", "Q8_0"] + (["Q4_K", "Q6_K"] if kind == "layer" else ["Q4_K_M", "F16"])
        hidden = 256 * _log(rng, 2, 24 if kind == "layer" else 16)
        c.update(type=rng.choice(types), hidden=hidden, kv=hidden // rng.choice([1, 4, 8]) // 16 * 16,
                 ffn=256 * int(hidden * rng.uniform(2, 4) / 256))
        if kind == "blayer":
            c["batch"] = rng.randint(2, 16)
    elif kind == "linear":
        t = rng.choice(sorted(TYPES))
        cols = _cols(rng, t)
        c.update(type=t, rows=min(_log(rng, 1, 32000), max(1, (400 << 20) // (4 * cols))), cols=cols,
                 acc=rng.random() < 0.3)
    elif kind == "batch":
        t = rng.choice(sorted(TYPES))
        cols = _cols(rng, t, hi=14336)
        c.update(type=t, rows=min(_log(rng, 1, 32000), max(1, (200 << 20) // (4 * cols))), cols=cols,
                 batch=rng.randint(2, 16))
    elif kind == "head":
        c.update(type=rng.choice(["Q6_K", "Q8_0", "Q4_K", "F16"]), vocab=_log(rng, 256, 64000),
                 dim=256 * rng.randint(1, 32), ids=_log(rng, 1, 512))
    elif kind == "attention":
        kvh = rng.choice([1, 2, 4, 8])
        c.update(heads=kvh * rng.choice([1, 2, 3, 4, 8]), kv_heads=kvh, hd=rng.choice([32, 64, 96, 128]),
                 seq=_log(rng, 1, 16384), layer=rng.randint(0, 1))
    else:
        t = rng.choice(["Q8_0", "Q4_0", "Q4_1", "F16", "F32"])
        cols = 32 * max(1, _log(rng, 32, 14336) // 32) if t[0] == "Q" else _log(rng, 32, 14336)
        c.update(type=t, rows=min(_log(rng, 1, 16000), max(1, (200 << 20) // (4 * cols))), cols=cols)
    return c


# ---- inputs -----------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _f16_bytes(v):
    return v.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _weights(t, rows, cols, g):
    """A packed rows x cols matrix of type t as uint8 (rows, row bytes), values as host/vbs_synth.c makes them."""
    e, bb = V.GEOMETRY[TYPES[t]]
    n = rows * (cols // e)
    if t == "F32":
        return torch.randn(rows, cols, generator=g, device=DEV).view(torch.uint8)
    if t == "F16":
        return torch.randn(rows, cols, generator=g, device=DEV, dtype=torch.float16).view(torch.uint8)
    words = torch.randint(-2**63, 2**63 - 1, ((n * bb + 7) // 8,), generator=g, device=DEV, dtype=torch.int64)
    b = words.view(torch.uint8)[:n * bb].reshape(n, bb)

    def scale():
        return _f16_bytes(torch.randn(n, generator=g, device=DEV).abs() * 0.01)

    if t == "Q6_K":
        b[:, 192:208] = b[:, 192:208] % 64 - 32  # (wraps to int8 -32 .. 31)
        b[:, 208:210] = scale()
    elif t == "LNS8":
        b[:, :32] %= 12
        b[:, 32:36] = (torch.rand(n, 1, generator=g, device=DEV) / 256).view(torch.uint8)
    else:
        if t == "Q8_0":
            b[b == 128] = 0  # quants are -127 .. 127
        b[:, 0:2] = scale()
        if t == "Q4_1":
            b[:, 2:4] = _f16_bytes(torch.randn(n, generator=g, device=DEV) * 0.01)
        if t == "Q4_K":
            b[:, 2:4] = scale()
    return b.reshape(rows, -1)


def _randn(g, *shape, scale=1.0, offset=0.0):
    return torch.randn(*shape, generator=g, device=DEV) * scale + offset


def _shapes(geo):
    """(rows, cols) of the seven matrices of a layer."""
    H, F, nq, nkv, hd, _ = geo
    return {"q": (nq * hd, H), "k": (nkv * hd, H), "v": (nkv * hd, H), "o": (H, nq * hd), "gate": (F, H),
            "up": (F, H), "down": (H, F)}


def _set_shapes(case):
    """The matrices of a matvec layer set."""
    H = case["hidden"]
    return _shapes((H, case["ffn"], H // 16, case["kv"] // 16, 16, 0))


def _mix(t, role):
    return ("Q6_K" if role in ("down", "head", "embd") else "Q4_K") if t == "Q4_K_M" else t


class _Held:
    """A state whose decoder or graph goes with it."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        for f in self.__dict__.get("close", ()):
            f()


_dev = None


def _lib():
    global _dev
    if _dev is None:
        d = V.DeviceLib()
        if not d.init():
            raise RuntimeError(d.error())
        _dev = d
    return _dev


def _ptr_array(ts):
    return (C.c_void_p * len(ts))(*[t.data_ptr() for t in ts])


def _model(geo, layers, pos, g, batch=1, max_ctx=None):
    """Weights, norms and caches of a Q4_K_M model on the device and the library's description of them."""
    H, F, nq, nkv, hd, vocab = geo
    ctx = max_ctx or pos + 8
    m = {"embd": _weights("Q6_K", vocab, H, g), "head": _weights("Q6_K", vocab, H, g),
         "out_norm": _randn(g, H, scale=0.1, offset=1.0),
         "attn_norm": [_randn(g, H, scale=0.1, offset=1.0) for _ in range(layers)],
         "ffn_norm": [_randn(g, H, scale=0.1, offset=1.0) for _ in range(layers)],
         "w": [_weights(_mix("Q4_K_M", r), *_shapes(geo)[r], g) for _ in range(layers) for r in ROLES]}
    shape = (batch, layers, ctx, nkv * hd)
    m["kc"] = torch.randn(*shape, generator=g, device=DEV, dtype=torch.float16).view(torch.int16)
    m["vc"] = torch.randn(*shape, generator=g, device=DEV, dtype=torch.float16).view(torch.int16)
    wtype = np.array([TYPES[_mix("Q4_K_M", r)] for _ in range(layers) for r in ROLES], np.int32)
    keep = (wtype, _ptr_array(m["attn_norm"]), _ptr_array(m["ffn_norm"]), _ptr_array(m["w"]))
    m["view"] = V.Gfx950ModelStruct(layers, H, F, nq, nkv, hd, vocab, ctx, THETA, EPS, V.Q6_K,
                                    m["embd"].data_ptr(), m["out_norm"].data_ptr(), V.Q6_K, m["head"].data_ptr(),
                                    C.addressof(keep[1]), C.addressof(keep[2]), wtype.ctypes.data,
                                    C.addressof(keep[3]), m["kc"].data_ptr(), m["vc"].data_ptr())
    m["keep"] = keep
    return m


class _HostModel:
    """What V.Decoder takes of a model: packed weights in host memory."""

    def __init__(self, case, g):
        H, F, nq, nkv, hd, vocab = geo = _ops_geo(case)
        L, mix = case["layers"], case["mix"]
        host = lambda t: np.ascontiguousarray(t.cpu().numpy())  # noqa: E731
        self.cfg = {"vocab": vocab, "n_layers": L, "n_kv_heads": nkv, "head_dim": hd}
        self.embd = host(_weights(_mix(mix, "embd"), vocab, H, g))
        self.head = host(_weights(_mix(mix, "head"), vocab, H, g))
        self.out_norm = host(_randn(g, H, scale=0.1, offset=1.0))
        self.norms = [host(_randn(g, H, scale=0.1, offset=1.0)) for _ in range(2 * L)]
        self.w = [host(_weights(_mix(mix, r), *_shapes(geo)[r], g)) for _ in range(L) for r in ROLES]
        kv = (L, case["pos"], nkv * hd)
        self.kc = host(torch.randn(*kv, generator=g, device=DEV, dtype=torch.float16).view(torch.int16)).view(np.uint16)
        self.vc = host(torch.randn(*kv, generator=g, device=DEV, dtype=torch.float16).view(torch.int16)).view(np.uint16)
        self.wtype = np.array([TYPES[_mix(mix, r)] for _ in range(L) for r in ROLES], np.int32)
        ptrs = lambda a: (C.c_void_p * len(a))(*[x.ctypes.data for x in a])  # noqa: E731
        self.pa, self.pf, self.pw = ptrs(self.norms[:L]), ptrs(self.norms[L:]), ptrs(self.w)
        self.struct = V.DecodeModelStruct(L, H, F, nq, nkv, hd, vocab, case["pos"] + 8, THETA, EPS,
                                          TYPES[_mix(mix, "embd")], self.embd.ctypes.data, self.out_norm.ctypes.data,
                                          TYPES[_mix(mix, "head")], self.head.ctypes.data, C.addressof(self.pa),
                                          C.addressof(self.pf), self.wtype.ctypes.data, C.addressof(self.pw))

    def decode_struct(self):
        return self.struct


def _ops_geo(case):
    return tuple(case[k] for k in ("hidden", "ffn", "heads", "kv_heads", "hd", "vocab"))


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g, k = _gen(seed), case["kind"]
    if k == "decode":
        m = _model(GEO[case["geo"]], case["layers"], case["pos"], g)
        m["token"] = int(torch.randint(0, GEO[case["geo"]][5], (1,), generator=g, device=DEV))
        return m
    if k == "bdecode":
        m = _model(GEO[case["geo"]], case["layers"], case["pos"], g, batch=case["batch"])
        m["tokens"] = torch.randint(0, GEO[case["geo"]][5], (case["batch"],), generator=g, device=DEV).cpu().numpy().astype(np.uint32)
        # each sequence at a position of its own, the longest at `pos`
        m["pos"] = np.array([max(0, case["pos"] - b * (case["pos"] // 16)) for b in range(case["batch"])], np.uint32)
        return m
    if k in ("layer", "blayer"):
        n = case.get("batch", 1)
        sh = _set_shapes(case)
        w = {r: _weights(_mix(case["type"], r), *sh[r], g) for r in ROLES}
        return {"w": w, "x": {c: _randn(g, n, c) for c in sorted({c for _, c in sh.values()})},
                "y": {r: torch.zeros(n, sh[r][0], device=DEV) for r in ROLES}}
    if k in ("linear", "batch"):
        n = case.get("batch", 1)
        return {"w": _weights(case["type"], case["rows"], case["cols"], g), "x": _randn(g, n, case["cols"]),
                "y": _randn(g, n, case["rows"])}
    if k == "head":
        return {"w": _weights(case["type"], case["vocab"], case["dim"], g), "x": _randn(g, case["dim"]),
                "ids": torch.randint(0, case["vocab"], (case["ids"],), generator=g, device=DEV, dtype=torch.int32),
                "y": torch.zeros(case["vocab"], device=DEV), "rows": torch.zeros(case["ids"], case["dim"], device=DEV)}
    if k == "attention":
        kvd = case["kv_heads"] * case["hd"]
        shape = (case["layer"] + 1, case["seq"] + 7, kvd)
        return {"q": _randn(g, case["heads"] * case["hd"]), "out": torch.zeros(case["heads"] * case["hd"], device=DEV),
                "kc": torch.randn(*shape, generator=g, device=DEV, dtype=torch.float16),
                "vc": torch.randn(*shape, generator=g, device=DEV, dtype=torch.float16)}
    if k == "hot":
        rows, cols = case["rows"], case["cols"]
        nb = max(1, cols // 32)
        return {"w": _weights(case["type"], rows, cols, g), "x": _randn(g, cols),
                "xq": torch.zeros(cols, dtype=torch.int8, device=DEV), "qd": torch.zeros(nb, device=DEV),
                "qsum": torch.zeros(nb, device=DEV), "y": torch.zeros(rows, device=DEV)}
    raise ValueError(k)


def prepare(case, seed):
    dev, k = _lib(), case["kind"]
    if k == "ops":
        be = V.gfx950_backend()
        if not be.init():
            raise RuntimeError(be.last_error())
        m = _HostModel(case, _gen(seed))
        d = V.Decoder(V.load_host(), be, m)
        if case["pos"]:
            d.load_kv(m.kc, m.vc, case["pos"])
        return _Held(case=case, d=d, model=m, token=int(seed) % case["vocab"], close=(d.close,))
    s = _Held(case=case, dev=dev, **_inputs(case, seed))
    torch.cuda.synchronize()
    if k in ("decode", "bdecode"):
        h = C.c_void_p()
        if k == "decode":
            dev.check(dev._decoder_create(C.addressof(s.view), 16, C.byref(h)), "decoder_create")
            s.close = (lambda: dev._decoder_destroy(h.value),)
        else:
            dev.check(dev._bdecoder_create(C.addressof(s.view), case["batch"], s.kc.stride(0), 16, C.byref(h)),
                      "bdecoder_create")
            s.close = (lambda: dev._bdecoder_destroy(h.value),)
        s.h = h.value
    elif k in ("layer", "blayer"):
        # one graph for the set's launches, as bench.py keeps one per weight copy
        hip, stream = V.Hip(), dev.stream()
        _enqueue(s)
        dev.sync()
        graph = hip.capture(stream, lambda: _enqueue(s))
        s.hip, s.stream, s.graph = hip, stream, graph
        s.close = (lambda: hip.destroy(graph),)
    return s


GROUPS = (("q", "k", "v"), ("o",), ("gate", "up"), ("down",))


def _enqueue(s):
    sh, t = _set_shapes(s.case), s.case["type"]
    if s.case["kind"] == "layer":
        for r in ROLES:
            rows, cols = sh[r]
            s.dev.linear(TYPES[t], s.w[r].data_ptr(), s.x[cols].data_ptr(), s.y[r].data_ptr(), cols, rows)
        return
    for group in GROUPS:
        cols, rows = sh[group[0]][1], [sh[r][0] for r in group]
        s.dev.linear_batch_multi(TYPES[_mix(t, group[0])], [s.w[r].data_ptr() for r in group], rows,
                                 s.x[cols].data_ptr(), cols, [s.y[r].data_ptr() for r in group], rows, cols,
                                 s.case["batch"])


def run(s):
    c = s.case
    k = c["kind"]
    if k == "ops":
        return s.d.step(s.token, c["pos"])
    dev = s.dev
    if k == "decode":
        logits = np.empty(GEO[c["geo"]][5], np.float32)
        dev.check(dev._decoder_step(s.h, s.token, c["pos"], logits.ctypes.data), "decoder_step")
        return {"logits": logits, "k": s.kc[0, :, c["pos"]], "v": s.vc[0, :, c["pos"]]}
    if k == "bdecode":
        logits = np.empty((c["batch"], GEO[c["geo"]][5]), np.float32)
        dev.check(dev._bdecoder_step(s.h, s.tokens.ctypes.data, s.pos.ctypes.data, logits.ctypes.data),
                  "bdecoder_step")
        return {"logits": logits, "k": s.kc[0, :, c["pos"]], "v": s.vc[0, :, c["pos"]]}
    if k in ("layer", "blayer"):
        s.hip.launch(s.graph, s.stream)
        return [s.y[r] for r in ROLES]
    if k == "linear":
        dev.linear(TYPES[c["type"]], s.w.data_ptr(), s.x.data_ptr(), s.y.data_ptr(), c["cols"], c["rows"],
                   accumulate=c["acc"])
        return s.y
    if k == "batch":
        dev.linear_batch(TYPES[c["type"]], s.w.data_ptr(), s.x.data_ptr(), c["cols"], s.y.data_ptr(), c["rows"],
                         c["cols"], c["rows"], c["batch"])
        return s.y
    if k == "head":
        t = TYPES[c["type"]]
        dev.linear(t, s.w.data_ptr(), s.x.data_ptr(), s.y.data_ptr(), c["dim"], c["vocab"])
        dev.dequant_rows(t, s.w.data_ptr(), s.ids.data_ptr(), c["ids"], c["dim"], s.rows.data_ptr())
        return [s.y, s.rows]
    if k == "attention":
        dev.attention(s.q.data_ptr(), s.kc.data_ptr(), s.vc.data_ptr(), s.out.data_ptr(), c["seq"], c["layer"],
                      s.kc.shape[1], c["heads"], c["kv_heads"], c["hd"], 1.0 / math.sqrt(c["hd"]))
        return s.out
    if c["type"] in ("Q8_0", "Q4_0", "Q4_1"):
        dev.quantize_q8(s.x.data_ptr(), c["cols"], s.xq.data_ptr(), s.qd.data_ptr(), s.qsum.data_ptr())
        dev.hot_matvec(TYPES[c["type"]], s.w.data_ptr(), c["rows"], c["cols"], s.xq.data_ptr(), s.qd.data_ptr(),
                       s.qsum.data_ptr(), s.y.data_ptr())
    else:
        dev.hot_matvec(TYPES[c["type"]], s.w.data_ptr(), c["rows"], c["cols"], s.x.data_ptr(), 0, 0, s.y.data_ptr())
    return s.y


# ---- what a pass needs ----------------------------------------------------------------------

def _step_work(geo, mix, layers, positions):
    H, F, nq, nkv, hd, vocab = geo
    n = len(positions)
    mats = [(_mix(mix, r), *s) for r, s in _shapes(geo).items()] * layers + [(_mix(mix, "head"), vocab, H)]
    w = sum(V.row_bytes(TYPES[t], c) * r for t, r, c in mats) + 4 * H * (2 * layers + 1)
    kv = sum(2 * 2 * layers * (p + 1) * nkv * hd for p in positions)
    flops = 2 * n * sum(r * c for _, r, c in mats) + sum(4 * layers * (p + 1) * nq * hd for p in positions)
    return {"bytes": w + kv + n * (V.row_bytes(TYPES[_mix(mix, "embd")], H) + 4 * vocab), "flops": flops}


def work(case):
    k = case["kind"]
    if k == "ops":
        return _step_work(_ops_geo(case), case["mix"], case["layers"], [case["pos"]])
    if k == "decode":
        return _step_work(GEO[case["geo"]], "Q4_K_M", case["layers"], [case["pos"]])
    if k == "bdecode":
        return _step_work(GEO[case["geo"]], "Q4_K_M", case["layers"],
                          [max(0, case["pos"] - b * (case["pos"] // 16)) for b in range(case["batch"])])
    n = case.get("batch", 1)
    if k in ("layer", "blayer"):
        sh = _set_shapes(case)
        return {"bytes": sum(V.row_bytes(TYPES[_mix(case["type"], r)], c) * m + 4 * n * (m + c) for r, (m, c) in sh.items()),
                "flops": sum(2 * n * m * c for m, c in sh.values())}
    if k in ("linear", "batch"):
        m, c = case["rows"], case["cols"]
        return {"bytes": V.row_bytes(TYPES[case["type"]], c) * m + 4 * n * (c + m * (2 if case.get("acc") else 1)),
                "flops": 2 * n * m * c}
    if k == "head":
        rb = V.row_bytes(TYPES[case["type"]], case["dim"])
        return {"bytes": rb * (case["vocab"] + case["ids"]) + 4 * (case["dim"] + case["vocab"] + case["ids"] * (1 + case["dim"])),
                "flops": 2 * case["vocab"] * case["dim"]}
    if k == "attention":
        return {"bytes": 4 * case["seq"] * case["kv_heads"] * case["hd"] + 8 * case["heads"] * case["hd"],
                "flops": 4 * case["seq"] * case["heads"] * case["hd"]}
    m, c = case["rows"], case["cols"]
    return {"bytes": V.row_bytes(TYPES[case["type"]], c) * m + 4 * c + 4 * m, "flops": 2 * m * c}


def tolerance(case):
    k = case["kind"]
    if k == "hot":
        return "exact"  # its sums have one defined order
    if k in ("decode", "bdecode"):
        # f32 sums through the layers (logits 4 to 8e-7 off in 64 bits); a cache value may round to the next f16
        return {"rel": 5e-6, "max": 5e-5, "differ": 4e-3}
    if k == "ops":
        return {"rel": 5e-6, "max": 5e-5}
    return {"rel": 2e-6, "max": 2e-5}  # f32 sums (1 to 5e-7 off in 64 bits)


# ---- the same in 64 bits -----------------------------------------------------------------------

def _half(b):
    return b.contiguous().view(torch.float16).to(torch.float64)


def _nibbles(q):
    return torch.cat([q & 15, q >> 4], -1)


def _deq(t, w, cols):
    """The values of packed rows w (uint8) in float64."""
    if t == "F32":
        return w.view(torch.float32).to(torch.float64)
    if t == "F16":
        return w.view(torch.float16).to(torch.float64)
    rows = w.shape[0]
    e, bb = V.GEOMETRY[TYPES[t]]
    b = w.reshape(rows, cols // e, bb)
    if t == "Q8_0":
        v = _half(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8)
    elif t == "Q4_0":
        v = _half(b[..., :2]) * (_nibbles(b[..., 2:]).to(torch.float64) - 8)
    elif t == "Q4_1":
        v = _half(b[..., :2]) * _nibbles(b[..., 4:]) + _half(b[..., 2:4])
    elif t == "LNS8":
        v = torch.exp2(b[..., :32].to(torch.float64)) * b[..., 32:].contiguous().view(torch.float32).to(torch.float64)
    elif t == "Q4_K":
        s = b[..., 4:16]
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | (s[..., 0:4] >> 6 << 4)], -1)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | (s[..., 4:8] >> 6 << 4)], -1)
        q = b[..., 16:].reshape(rows, -1, 4, 32)
        q = torch.stack([q & 15, q >> 4], -2).reshape(rows, -1, 8, 32)
        v = (_half(b[..., 0:2]) * sc).unsqueeze(-1) * q - (_half(b[..., 2:4]) * mn).unsqueeze(-1)
    else:  # Q6_K: halves of 128, each four quarters of 32
        ql, qh = b[..., :128].reshape(rows, -1, 2, 2, 32), b[..., 128:192].reshape(rows, -1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], -2)
        hi = torch.cat([qh >> 2 * i & 3 for i in range(4)], -2)
        q = (lo | hi << 4).to(torch.int8) - 32
        v = (_half(b[..., 208:]) * b[..., 192:208].contiguous().view(torch.int8)).unsqueeze(-1) * q.reshape(rows, -1, 16, 16)
    return v.reshape(rows, cols)


def _matvec(t, w, x):
    """x (..., cols) times the packed matrix's transpose, in float64, some rows at a time."""
    cols, step = x.shape[-1], max(1, (1 << 27) // x.shape[-1])
    return torch.cat([x @ _deq(t, w[i:i + step], cols).T.contiguous() for i in range(0, w.shape[0], step)], -1)


def _attend(q, k, v, scale):
    """q (heads, hd), k and v (positions, kv heads, hd): softmax(q k) v, in float64."""
    group = q.shape[0] // k.shape[1]
    p = torch.softmax((q.reshape(k.shape[1], group, -1) @ k.permute(1, 2, 0).contiguous()) * scale, -1)
    return (p @ v.permute(1, 0, 2).contiguous()).reshape(-1)


def _step64(geo, mix, m, kc, vc, token, pos):
    """Logits of one token step and the K and V rows it stores; kc, vc (layers, positions, kv dim) f16."""
    H, F, nq, nkv, hd, vocab = geo
    f64 = torch.float64

    def norm(x, w):
        return x / torch.sqrt((x * x).mean() + EPS) * w.to(f64)

    angle = pos * THETA ** (-torch.arange(0, hd, 2, device=DEV, dtype=f64) / hd)
    cos, sin = torch.cos(angle), torch.sin(angle)

    def rope(v):
        a, b = v.reshape(-1, hd // 2, 2).unbind(-1)
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(-1)

    x = _deq(_mix(mix, "embd"), m["embd"][token:token + 1], H)[0]
    ks, vs = [], []
    for layer in range(kc.shape[0]):
        w = dict(zip(ROLES, m["w"][7 * layer:7 * layer + 7]))
        mv = lambda r, a: _matvec(_mix(mix, r), w[r], a)  # noqa: E731
        n = norm(x, m["attn_norm"][layer])
        q, k, v = rope(mv("q", n)), rope(mv("k", n)).half(), mv("v", n).half()
        ks.append(k)
        vs.append(v)
        full = lambda c, r: torch.cat([c[layer, :pos], r[None]]).to(f64).reshape(pos + 1, nkv, hd)  # noqa: E731
        x = x + mv("o", _attend(q.reshape(nq, hd), full(kc, k), full(vc, v), 1.0 / math.sqrt(hd)))
        n = norm(x, m["ffn_norm"][layer])
        x = x + mv("down", torch.nn.functional.silu(mv("gate", n)) * mv("up", n))
    return _matvec(_mix(mix, "head"), m["head"], norm(x, m["out_norm"])), torch.stack(ks), torch.stack(vs)


def exact(case, seed):
    k, f64 = case["kind"], torch.float64
    if k == "ops":
        h = _HostModel(case, _gen(seed))
        up = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
        L = case["layers"]
        m = {"embd": up(h.embd), "head": up(h.head), "out_norm": up(h.out_norm), "w": [up(a) for a in h.w],
             "attn_norm": [up(a) for a in h.norms[:L]], "ffn_norm": [up(a) for a in h.norms[L:]]}
        kc, vc = (up(a.view(np.int16)).view(torch.float16) for a in (h.kc, h.vc))
        return _step64(_ops_geo(case), case["mix"], m, kc, vc, int(seed) % case["vocab"], case["pos"])[0]
    s = _inputs(case, seed)
    if k == "decode":
        kc, vc = s["kc"][0].view(torch.float16), s["vc"][0].view(torch.float16)
        return {"logits": _step64(GEO[case["geo"]], "Q4_K_M", s, kc, vc, s["token"], case["pos"])[0], "k": None, "v": None}
    if k == "bdecode":
        got = [_step64(GEO[case["geo"]], "Q4_K_M", s, s["kc"][b].view(torch.float16), s["vc"][b].view(torch.float16),
                       int(s["tokens"][b]), int(s["pos"][b]))[0] for b in range(case["batch"])]
        return {"logits": torch.stack(got), "k": None, "v": None}
    if k in ("layer", "blayer"):
        sh = _set_shapes(case)
        return [_matvec(_mix(case["type"], r), s["w"][r], s["x"][sh[r][1]].to(f64)) for r in ROLES]
    if k in ("linear", "batch"):
        y = _matvec(case["type"], s["w"], s["x"].to(f64))
        return s["y"].to(f64) + y if case.get("acc") else y
    if k == "head":
        return [_matvec(case["type"], s["w"], s["x"].to(f64)),
                _deq(case["type"], s["w"][s["ids"].long()], case["dim"])]
    if k == "attention":
        n, hd = case["seq"], case["hd"]
        kv = [s[c][case["layer"], :n].to(f64).reshape(n, case["kv_heads"], hd) for c in ("kc", "vc")]
        return _attend(s["q"].to(f64).reshape(-1, hd), *kv, 1.0 / math.sqrt(hd))
    if case["type"] not in ("Q8_0", "Q4_0", "Q4_1"):
        return _matvec(case["type"], s["w"], s["x"].to(f64))
    # the table's own arithmetic: x as 32-element blocks of int8 with f16 scales (the quantised x is the definition)
    x = s["x"].reshape(-1, 32)
    d = x.abs().amax(1, keepdim=True) / 127
    v = x * (1 / d)
    q = torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v)).to(f64)  # half away from zero
    xq = (q * d.half().to(f64)).reshape(-1)
    if case["type"] != "Q4_1":
        return _matvec(case["type"], s["w"], xq)
    # min * sum is taken with a f16 sum: y = sum d q x + m h
    h = (q.sum(1, keepdim=True).float() * d).half().to(f64)
    w0 = s["w"].clone().reshape(-1, 20)
    m = _half(w0[:, 2:4]).reshape(case["rows"], -1)
    w0[:, 2:4] = 0
    return _matvec("Q4_1", w0.reshape(case["rows"], -1), xq) + m @ h.reshape(-1)
