"""The workloads this backend is timed on, through its public entry points.

A case names one kind of call and its sizes:

  matvec     `calls` mat-vecs (si_hip_gemv) called one by one without a plan:
             projections between other work of the caller, each its own weights
  products   a recorded plan of plain mat-vecs, `layers` copies of the listed
             weight shapes in order: the projections of a decode step
  chain      a recorded plan of a decoder's projections as the decode step
             fuses them: RMSNorm into qkv and gate/up, SwiGLU rows, residuals
             added by o and down, each product reading the one before
  prefill    a recorded plan of batched products Y = X . W^T at `m` prompt
             tokens of bf16 activations
  batch      a recorded plan of whole decoder layers of the 16-row prefill
             batch: norms, projections, rotary + cache append, causal
             attention, SwiGLU, rows `valid` of 16 live from position `start`
  attention  a recorded plan of one new token's attention per layer over the
             decode step's own fp16 cache layout (rotary and append included)
  gqa        grouped-query attention over [context][kv_heads][head] caches
  phi4       one token of a Phi-4-shaped model through its decode session
  rwkv7      one token of an RWKV-7-shaped model through its decode session

Weights are random GGUF blocks with the distributions of the benchmark
(synth_blocks), made on the GPU; activations are N(0, 1).
"""
import math

import numpy as np
import torch

from sharpinference_amd import native, phi4, rwkv7

FORMATS = {"q8_0": native.Q8_0, "q4_0": native.Q4_0, "q4_k": native.Q4_K, "f16": native.F16, "f32": native.F32}
BLOCK = {"q8_0": 32, "q4_0": 32, "q4_k": 256, "f16": 1, "f32": 1}
EPS = 1e-5
LAYER = "5120x3072,3072x3072,16384x3072,3072x8192"   # qkv, o, gate/up, down of the benchmark's decoder layer
F64 = torch.float64


def listed():
    return [
        # the smallest calls: the three receptance / key / value projections of an RWKV-7 layer, bound by call and launch
        {"name": "matvec_small", "kind": "matvec", "fmt": "q8_0", "rows": 2048, "cols": 2048, "calls": 3},
        # projections of a width outside the models built in, with a ragged row count
        {"name": "matvec_any_width", "kind": "matvec", "fmt": "q4_k", "rows": 5001, "cols": 11008, "calls": 2},
        # decode: the benchmark's Q4_0 layer set, enough layers to stream from HBM
        {"name": "decode_products", "kind": "products", "fmt": "q4_0", "shapes": LAYER, "layers": 12},
        # decode in the storage of the reference's own model (F16), fused as the decode step fuses it
        {"name": "decode_chain_f16", "kind": "chain", "fmt": "f16", "hidden": 3072, "qkv": 5120, "ffn": 8192,
         "layers": 4},
        # decode: one token of the whole Phi-4-mini-shaped model at 2048 cached tokens
        {"name": "decode_phi4", "kind": "phi4", "fmt": "q4_k", "layers": 32, "hidden": 3072, "heads": 24,
         "kv_heads": 8, "ffn": 8192, "vocab": 200064, "capacity": 4096, "position": 2048},
        # decode: one token of the whole RWKV-7 1.5B-shaped model
        {"name": "decode_rwkv7", "kind": "rwkv7", "fmt": "q8_0", "layers": 24, "heads": 32, "ffn": 8192,
         "vocab": 65536},
        # prefill: a layer's products at the benchmark's 512 prompt tokens
        {"name": "prefill_512", "kind": "prefill", "fmt": "q4_0", "m": 512, "shapes": LAYER},
        # prefill: a long prompt in the decode benchmark's weight format
        {"name": "prefill_2048", "kind": "prefill", "fmt": "q4_k", "m": 2048, "shapes": LAYER},
        # prefill: a short prompt (a chat turn), ragged token count
        {"name": "prefill_33", "kind": "prefill", "fmt": "q8_0", "m": 33, "shapes": LAYER},
        # prefill by 16-row batches, the reference's prefill program: two whole layers in the middle of a prompt
        {"name": "batch_layers", "kind": "batch", "fmt": "q4_k", "layers": 2, "hidden": 3072, "heads": 24,
         "kv_heads": 8, "ffn": 8192, "context": 4096, "start": 1016, "valid": 16, "cache": "f16"},
        # decode attention at a long context, eight layers' caches
        {"name": "attention_long", "kind": "attention", "heads": 24, "kv_heads": 8, "rotary": 96, "capacity": 8192,
         "position": 8000, "layers": 8},
        # the reference's attention operator: FP32 caches, 64-value heads, eight query heads per KV head
        {"name": "gqa_f32_head64", "kind": "gqa", "heads": 32, "kv_heads": 4, "head": 64, "context": 4096,
         "position": 4000, "cache": "f32", "layers": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cols(rng, fmt, lo, hi):
    """Half the time a power-of-two-ish model width, else any whole number of blocks."""
    unit = BLOCK[fmt]
    if rng.random() < 0.5:
        return rng.choice([c for c in (256, 512, 1024, 2048, 3072, 4096, 6144, 8192) if lo <= c <= hi])
    return max(1, _log(rng, lo, hi) // unit) * unit


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "products", "chain", "prefill", "prefill", "prefill", "batch", "batch",
                       "attention", "gqa", "phi4", "rwkv7"])
    quant = rng.choice(["q8_0", "q4_0", "q4_k"])
    fmt = rng.choice(["q8_0", "q4_0", "q4_k", "q4_k", "f16", "f32"])
    if kind == "matvec":
        return {"kind": kind, "fmt": fmt, "rows": _log(rng, 64, 24000), "cols": _cols(rng, fmt, 256, 14336),
                "calls": rng.randint(2, 4)}
    if kind == "products":
        shapes = ",".join("%dx%d" % (_log(rng, 256, 16384), _cols(rng, fmt, 512, 8192)) for _ in range(rng.randint(1, 4)))
        return {"kind": kind, "fmt": fmt, "shapes": shapes, "layers": rng.randint(1, 4)}
    if kind == "chain":
        hidden = rng.choice([1024, 2048, 3072, 4096])
        return {"kind": kind, "fmt": fmt, "hidden": hidden, "qkv": hidden + rng.choice([256, 1024, 2048, 2 * hidden]),
                "ffn": 256 * rng.randint(4, 40), "layers": rng.randint(1, 4)}
    if kind == "prefill":
        rows, cols = _log(rng, 64, 16384), _cols(rng, "q4_k" if fmt == "q4_k" else "q8_0", 256, 8192)
        m = min(_log(rng, 1, 2048), max(1, int(2e11 / (rows * cols))))
        return {"kind": kind, "fmt": fmt, "m": m, "shapes": "%dx%d" % (rows, cols)}
    if kind == "batch":
        kv = rng.choice([2, 4, 8])
        heads = kv * rng.randint(1, 4)
        context = _log(rng, 64, 8192)
        valid = rng.choice([16, rng.randint(1, 15)])
        return {"kind": kind, "fmt": fmt, "layers": rng.randint(1, 2), "hidden": 128 * heads, "heads": heads,
                "kv_heads": kv, "ffn": 256 * rng.randint(4, 40), "context": context,
                "start": rng.randint(0, context - valid), "valid": valid, "cache": rng.choice(["f16", "f32"])}
    if kind == "attention":
        kv = rng.choice([1, 2, 4, 8])
        capacity = _log(rng, 64, 16384)
        return {"kind": kind, "heads": kv * rng.randint(1, 4), "kv_heads": kv,
                "rotary": rng.choice([64, 96, 96, 128, 128, 40]), "capacity": capacity,
                "position": rng.randint(0, capacity - 1), "layers": rng.randint(1, 8)}
    if kind == "gqa":
        kv = rng.choice([1, 2, 4, 8])
        context = _log(rng, 64, 16384)
        return {"kind": kind, "heads": kv * rng.choice([1, 2, 3, 4, 6, 8]), "kv_heads": kv,
                "head": rng.choice([64, 128, 128, 256]), "context": context, "position": rng.randint(0, context - 1),
                "cache": rng.choice(["f16", "f32"]), "layers": rng.randint(1, 8)}
    if kind == "phi4":
        kv = rng.choice([2, 4, 8])
        heads = kv * rng.choice([c for c in (1, 2, 3, 4) if 128 * kv * c in (1024, 2048, 3072, 4096)])
        capacity = _log(rng, 256, 4096)
        return {"kind": kind, "fmt": quant, "layers": rng.randint(1, 12), "hidden": 128 * heads, "heads": heads,
                "kv_heads": kv, "ffn": rng.choice([2048, 3072, 4096, 6144, 8192]), "vocab": _log(rng, 1000, 100000),
                "capacity": capacity, "position": rng.randint(0, capacity - 1)}
    heads = rng.choice([16, 32, 48])
    return {"kind": kind, "fmt": quant if quant != "q4_k" else "q8_0", "layers": rng.randint(1, 12), "heads": heads,
            "ffn": 4 * 64 * heads if heads < 48 else 8192, "vocab": _log(rng, 1000, 65536)}


# ---- inputs -------------------------------------------------------------------------------

def _shapes(case):
    return [tuple(int(v) for v in s.split("x")) for s in case["shapes"].split(",")]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _norm_weight(g, n):
    return 1.0 + 0.1 * _randn(g, n)


def _half_bytes(v):
    return v.half().view(torch.uint8).reshape(-1, 2)


def _blocks(g, fmt, rows, cols, sigma=0.02):
    """[rows, cols] random weights in their GGUF bytes (uint8)."""
    if fmt in ("f16", "f32"):
        w = _randn(g, rows, cols).mul_(sigma)
        return (w.half() if fmt == "f16" else w).view(torch.uint8).reshape(-1)
    nb = rows * cols // BLOCK[fmt]

    def ints(lo, hi, *shape):
        return torch.randint(lo, hi, shape, device="cuda", generator=g, dtype=torch.uint8)

    if fmt == "q8_0":
        out = torch.empty(nb, 34, device="cuda", dtype=torch.uint8)
        out[:, :2] = _half_bytes(_randn(g, nb).abs() * (sigma / 127))
        out[:, 2:] = torch.randint(-127, 128, (nb, 32), device="cuda", generator=g, dtype=torch.int8).view(torch.uint8)
    elif fmt == "q4_0":
        out = torch.empty(nb, 18, device="cuda", dtype=torch.uint8)
        out[:, :2] = _half_bytes(_randn(g, nb).abs() * (sigma / 8))
        out[:, 2:] = ints(0, 255, nb, 16)
    else:
        out = torch.empty(nb, 144, device="cuda", dtype=torch.uint8)
        out[:, 0:2] = _half_bytes(_randn(g, nb).abs() * (sigma / 504))
        out[:, 2:4] = _half_bytes(_randn(g, nb).abs() * (sigma / 63))
        sc, m = ints(0, 64, nb, 8), ints(0, 64, nb, 8)
        out[:, 4:8] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
        out[:, 8:12] = m[:, :4] | ((m[:, 4:] >> 4) << 6)
        out[:, 12:16] = (sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)
        out[:, 16:] = ints(0, 255, nb, 128)
    return out.reshape(-1)


def _weights(g, fmt, shapes):
    return [_blocks(g, fmt, r, c) for r, c in shapes]


def _layer_shapes(case):
    h, kv = case["hidden"], 128 * case["kv_heads"]
    return [(h + 2 * kv, h), (h, h), (2 * case["ffn"], h), (h, case["ffn"])]


def _inputs(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "matvec":
        return {"w": [_blocks(g, case["fmt"], case["rows"], case["cols"]) for _ in range(case["calls"])],
                "x": _randn(g, case["cols"])}
    if kind == "products":
        shapes = _shapes(case)
        return {"w": [_weights(g, case["fmt"], shapes) for _ in range(case["layers"])],
                "x": {c: _randn(g, c) for c in sorted({c for _, c in shapes})}}
    if kind == "chain":
        h, f = case["hidden"], case["ffn"]
        shapes = [(case["qkv"], h), (h, h), (2 * f, h), (h, f)]
        return {"w": [_weights(g, case["fmt"], shapes) for _ in range(case["layers"])], "h": _randn(g, h),
                "norms": [[_norm_weight(g, h), _norm_weight(g, h)] for _ in range(case["layers"])]}
    if kind == "prefill":
        shapes = _shapes(case)
        return {"w": _weights(g, case["fmt"], shapes),
                "x": {c: _randn(g, case["m"], c).bfloat16() for c in sorted({c for _, c in shapes})}}
    if kind == "batch":
        n, h, kvw = case["layers"], case["hidden"], 128 * case["kv_heads"]
        dt = torch.float16 if case["cache"] == "f16" else torch.float32
        return {"w": [_weights(g, case["fmt"], _layer_shapes(case)) for _ in range(n)], "h": _randn(g, 16, h),
                "norms": [[_norm_weight(g, h), _norm_weight(g, h)] for _ in range(n)], "out_norm": _norm_weight(g, h),
                "k": _randn(g, n, case["context"], kvw).to(dt), "v": _randn(g, n, case["context"], kvw).to(dt),
                "freq": _frequencies(96), "control": torch.tensor([case["start"], case["valid"]], device="cuda",
                                                                  dtype=torch.int32)}
    if kind == "attention":
        n, kv = case["layers"], case["kv_heads"]
        return {"qkv": _randn(g, n, (case["heads"] + 2 * kv) * 128),
                "k": _randn(g, n, kv, case["capacity"], 128).half(), "v": _randn(g, n, kv, case["capacity"], 128).half(),
                "position": torch.tensor([case["position"]], device="cuda", dtype=torch.int32)}
    if kind == "gqa":
        n, d = case["layers"], case["head"]
        dt = torch.float16 if case["cache"] == "f16" else torch.float32
        return {"q": _randn(g, n, case["heads"] * d), "k": _randn(g, n, case["context"], case["kv_heads"] * d).to(dt),
                "v": _randn(g, n, case["context"], case["kv_heads"] * d).to(dt),
                "position": torch.tensor([case["position"]], device="cuda", dtype=torch.int32)}
    if kind == "phi4":
        n, h = case["layers"], case["hidden"]
        return {"w": [_weights(g, case["fmt"], _layer_shapes(case)) for _ in range(n)],
                "embed": _blocks(g, "q8_0", case["vocab"], h), "head": _blocks(g, "q8_0", case["vocab"], h),
                "norms": [[_norm_weight(g, h), _norm_weight(g, h)] for _ in range(n)], "out_norm": _norm_weight(g, h),
                "kv": [[_randn(g, case["kv_heads"], case["position"], 128).half() for _ in range(2)] for _ in range(n)],
                "token": int(seed) * 7919 % case["vocab"]}
    d = 64 * case["heads"]
    cfg = _rwkv_config(case)
    distinct = min(4, case["layers"])

    def layer():
        out = {k: _blocks(g, case["fmt"], r, c) for k, (r, c) in cfg.matrix_shapes(1).items()}
        for k in ("ln1_weight", "ln2_weight", "lnx_weight", "k_k"):
            out[k] = _norm_weight(g, d)
        for k in ("ln1_bias", "ln2_bias", "lnx_bias", "r_k"):
            out[k] = 0.1 * _randn(g, d)
        for k in ("w0", "a0", "v0"):
            out[k] = _randn(g, d)
        for k in ("k_a", "ffn_mix"):
            out[k] = torch.rand(d, device="cuda", generator=g)
        out["mix"] = torch.rand(6, d, device="cuda", generator=g)
        return out

    gen = [layer() for _ in range(distinct)]
    return {"layers": [gen[i % distinct] for i in range(case["layers"])], "embed": _blocks(g, "q8_0", case["vocab"], d),
            "head": _blocks(g, "q8_0", case["vocab"], d), "ln0": [_norm_weight(g, d), 0.1 * _randn(g, d)],
            "ln_out": [_norm_weight(g, d), 0.1 * _randn(g, d)],
            "state": [[_randn(g, d), _randn(g, d), 0.1 * _randn(g, case["heads"], 64, 64)] for _ in range(case["layers"])],
            "token": int(seed) * 7919 % case["vocab"]}


def _frequencies(rotary):
    i = torch.arange(rotary // 2, device="cuda", dtype=torch.float32)
    return 1.0 / torch.pow(torch.tensor(10000.0, device="cuda"), 2.0 * i / rotary)


def _phi4_config(case):
    return phi4.Phi4Config(layers=case["layers"], hidden=case["hidden"], heads=case["heads"],
                           kv_heads=case["kv_heads"], ffn=case["ffn"], vocab=case["vocab"], capacity=case["capacity"],
                           weight_format=FORMATS[case["fmt"]])


def _rwkv_config(case):
    return rwkv7.Rwkv7Config(layers=case["layers"], hidden=64 * case["heads"], heads=case["heads"], ffn=case["ffn"],
                             vocab=case["vocab"], weight_format=FORMATS[case["fmt"]])


# ---- the program --------------------------------------------------------------------------

_hip = None


def _context():
    """The program's one context."""
    global _hip
    if _hip is None:
        _hip = native.HipContext(0)
    return _hip


class _Owner:
    """Keeps a state's device memory and plan, and gives them back with the state."""

    def __init__(self, held=None):
        self.held = held
        self.plan = None
        self.session = None

    def __del__(self):
        _context().sync()
        if self.plan is not None:
            self.plan.destroy()
        if self.session is not None:
            self.session.close()


class _DeviceArray:
    """A library buffer as torch sees it (no copy); keeps its owner alive."""

    def __init__(self, owner, buffer, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (buffer.ptr, False),
                                         "version": 3}


def _tensor(owner, buffer, shape, typestr="<f4"):
    return torch.as_tensor(_DeviceArray(owner, buffer, shape, typestr), device="cuda")


def _resident(hip, tensor):
    """A library buffer holding the tensor's bytes."""
    b = hip.alloc(tensor.numel() * tensor.element_size())
    hip.copy(b.ptr, tensor.data_ptr(), b.nbytes)
    return b


def _empty(*shape):
    return torch.empty(*shape, device="cuda")


def prepare(case, seed):
    hip, kind = _context(), case["kind"]
    inp = _inputs(case, seed)
    torch.cuda.synchronize()
    owner = _Owner(inp)
    state = {"kind": kind, "owner": owner}
    fmt = FORMATS.get(case.get("fmt"))

    if kind == "matvec":
        state["out"] = [_empty(case["rows"]) for _ in inp["w"]]
        state["args"] = [(fmt, w.data_ptr(), inp["x"].data_ptr(), y.data_ptr(), case["rows"], case["cols"])
                         for w, y in zip(inp["w"], state["out"])]
        return state

    if kind == "products":
        shapes = _shapes(case)
        y = [[_empty(r) for r, _ in shapes] for _ in range(case["layers"])]

        def body():
            for ws, ys in zip(inp["w"], y):
                for (r, c), w, out in zip(shapes, ws, ys):
                    hip.gemv(fmt, w.data_ptr(), inp["x"][c].data_ptr(), out.data_ptr(), r, c)
        state["out"] = [out for ys in y for out in ys]

    elif kind == "chain":
        h, f, q = case["hidden"], case["ffn"], case["qkv"]
        bufs = [(_empty(q), _empty(h), _empty(f), _empty(h)) for _ in range(case["layers"])]
        owner.held = (inp, bufs)

        def body():
            x = inp["h"]
            for (wqkv, wo, wup, wdown), (n1, n2), (qkv, h1, act, h2) in zip(inp["w"], inp["norms"], bufs):
                p = lambda t: t.data_ptr()
                hip.gemv_batch([native.gemv_op(fmt, p(wqkv), p(x), p(qkv), q, h, xform=native.X_RMSNORM,
                                               norm_weight=p(n1), eps=EPS)])
                hip.gemv_batch([native.gemv_op(fmt, p(wo), p(qkv), p(h1), h, h, residual=p(x))])
                hip.gemv_batch([native.gemv_op(fmt, p(wup), p(h1), p(act), f, h, xform=native.X_RMSNORM,
                                               output=native.OUT_SWIGLU_ROWS, norm_weight=p(n2), eps=EPS)])
                hip.gemv_batch([native.gemv_op(fmt, p(wdown), p(act), p(h2), h, f, residual=p(h1))])
                x = h2
        state["out"] = [b for bs in bufs for b in bs]

    elif kind == "prefill":
        shapes, m = _shapes(case), case["m"]
        y = [_empty(m, r) for r, _ in shapes]

        def body():
            for (r, c), w, out in zip(shapes, inp["w"], y):
                hip.gemm_prefill(fmt, w.data_ptr(), inp["x"][c].data_ptr(), out.data_ptr(), m, r, c)
        state["out"] = y

    elif kind == "batch":
        state["out"], bufs, body = _batch_program(hip, case, inp)
        owner.held = (inp, bufs)

    elif kind == "attention":
        heads, kv, cap, n = case["heads"], case["kv_heads"], case["capacity"], case["layers"]
        out = _empty(n, heads * 128)
        ws = _empty(native.attention_workspace_bytes(heads, cap) // 4)
        owner.held = (inp, ws)
        args = [native.AttentionArgs(inp["qkv"][l].data_ptr(), inp["position"].data_ptr(), inp["k"][l].data_ptr(),
                                     inp["v"][l].data_ptr(), out[l].data_ptr(), ws.data_ptr(), heads, kv, 128,
                                     case["rotary"], cap, 10000.0, 1.0) for l in range(n)]

        def body():
            for a in args:
                hip.attention(a)
        at = case["position"]
        state["out"] = [out, inp["k"][:, :, at], inp["v"][:, :, at]]

    elif kind == "gqa":
        heads, kv, d, ctx, n = case["heads"], case["kv_heads"], case["head"], case["context"], case["layers"]
        out = _empty(n, heads * d)
        ws = _empty(native.gqa_workspace_bytes(heads, d, ctx) // 4)
        owner.held = (inp, ws)
        args = [native.GqaArgs(inp["q"][l].data_ptr(), inp["k"][l].data_ptr(), inp["v"][l].data_ptr(),
                               inp["position"].data_ptr(), out[l].data_ptr(), FORMATS[case["cache"]], heads, kv, d, ctx,
                               ws.data_ptr()) for l in range(n)]

        def body():
            for a in args:
                hip.grouped_query_attention(a)
        state["out"] = out

    elif kind == "phi4":
        up = lambda t: _resident(hip, t)
        per = lambda i: [up(ws[i]) for ws in inp["w"]]
        weights = phi4.Phi4Weights(embed=up(inp["embed"]), lm_head=up(inp["head"]), output_norm=up(inp["out_norm"]),
                                   attn_norm=[up(n[0]) for n in inp["norms"]], qkv=per(0), o=per(1),
                                   ffn_norm=[up(n[1]) for n in inp["norms"]], up=per(2), down=per(3))
        sess = phi4.Phi4DecodeSession(hip, _phi4_config(case), weights)
        row = 256 * case["capacity"]
        for layer, pair in zip(sess.layers, inp["kv"]):
            for name, src in zip(("k_cache", "v_cache"), pair):
                hip.fill_u32(layer[name].ptr, 0, layer[name].nbytes // 4)
                for head in range(case["kv_heads"]):
                    hip.copy(layer[name].ptr + head * row, src[head].data_ptr(), 256 * case["position"])
        hip.sync()
        owner.held, owner.session = None, sess
        state.update(session=sess, token=inp["token"], position=case["position"])
        last = sess.layers[-1]
        cache = lambda b: _tensor(owner, b, (case["kv_heads"], case["capacity"], 128), "<f2")[:, case["position"]]
        state["out"] = [_tensor(owner, sess.logits, (case["vocab"],)), cache(last["k_cache"]), cache(last["v_cache"])]
        return state

    else:
        host = lambda t: t.cpu().numpy()
        done = {}
        layers = []
        for layer in inp["layers"]:
            if id(layer) not in done:
                done[id(layer)] = {k: host(v) for k, v in layer.items()}
            layers.append(done[id(layer)])
        weights = rwkv7.Rwkv7Weights(embed=host(inp["embed"]), ln0_weight=host(inp["ln0"][0]),
                                     ln0_bias=host(inp["ln0"][1]), ln_out_weight=host(inp["ln_out"][0]),
                                     ln_out_bias=host(inp["ln_out"][1]), head=host(inp["head"]), layers=layers)
        sess = rwkv7.Rwkv7DecodeSession(hip, _rwkv_config(case), weights,
                                        [tuple(host(t) for t in s) for s in inp["state"]])
        owner.held, owner.session = None, sess
        state.update(session=sess, token=inp["token"])
        d = 64 * case["heads"]
        state["out"] = [_tensor(owner, sess.logits, (case["vocab"],))] + \
            [_tensor(owner, L["att_prev"], (d,)) for L in sess.layers] + \
            [_tensor(owner, L["wkv"], (case["heads"], 64, 64)) for L in sess.layers]
        return state

    owner.plan = hip.record(body)
    return state


def _batch_program(hip, case, inp):
    """Output tensors, scratch tensors and the launches of `layers` decoder layers over a 16-row batch."""
    B, h, f, heads, kv = 16, case["hidden"], case["ffn"], case["heads"], case["kv_heads"]
    qs, kvs, ctx, fmt, cache = 128 * heads, 128 * kv, case["context"], FORMATS[case["fmt"]], FORMATS[case["cache"]]
    n = case["layers"]
    zeros = lambda *s: torch.zeros(*s, device="cuda")   # rows past `valid` stay as they are
    normed, qkv, query, attn, proj = zeros(B, h), zeros(B, qs + 2 * kvs), zeros(B, qs), zeros(B, qs), zeros(B, h)
    gate_up, act, down = zeros(B, 2 * f), zeros(B, f), zeros(B, h)
    hidden = [inp["h"]] + [zeros(B, h) for _ in range(2 * n)]
    out = zeros(B, h)
    ws = zeros(native.batch_values_workspace_bytes(B, heads, ctx) // 4)
    torch.cuda.synchronize()
    p = lambda t: t.data_ptr()
    ctl = p(inp["control"])

    def body():
        for l in range(n):
            wqkv, wo, wup, wdown = inp["w"][l]
            n1, n2 = inp["norms"][l]
            at = hidden[2 * l]
            if l == 0:
                hip.batch_rms_norm(p(at), p(n1), ctl, p(normed), B, h, EPS)
            else:
                hip.batch_residual_rms_norm(p(hidden[2 * l - 1]), p(down), p(n1), ctl, p(at), p(normed), B, h, EPS)
            hip.batch_matvec(fmt, p(wqkv), p(normed), ctl, p(qkv), B, qs + 2 * kvs, h)
            k, v = inp["k"][l], inp["v"][l]
            hip.batch_rope_kv_write(native.BatchRopeArgs(p(qkv), ctl, p(inp["freq"]), p(query), p(k), p(v), cache, B, qs,
                                                         kvs, 128, 96, ctx, 1.0))
            hip.batch_gqa_attention(native.BatchAttentionArgs(p(query), 0, p(k), ctl, p(attn), p(ws), cache, B, heads, kv,
                                                              128, ctx), p(v))
            hip.batch_matvec(fmt, p(wo), p(attn), ctl, p(proj), B, h, h)
            hip.batch_residual_rms_norm(p(at), p(proj), p(n2), ctl, p(hidden[2 * l + 1]), p(normed), B, h, EPS)
            hip.batch_matvec(fmt, p(wup), p(normed), ctl, p(gate_up), B, 2 * f, h)
            hip.batch_swiglu(p(gate_up), ctl, p(act), B, f)
            hip.batch_matvec(fmt, p(wdown), p(act), ctl, p(down), B, h, f)
        hip.batch_residual_rms_norm(p(hidden[2 * n - 1]), p(down), p(inp["out_norm"]), ctl, p(hidden[2 * n]), p(out), B,
                                    h, EPS)

    rows = slice(case["start"], case["start"] + case["valid"])
    outs = [out, hidden[2 * n], inp["k"][:, rows], inp["v"][:, rows]]
    return outs, (normed, qkv, query, attn, proj, gate_up, act, down, hidden, ws), body


def run(state):
    kind = state["kind"]
    if kind == "matvec":
        hip = _context()
        for args in state["args"]:
            hip.gemv(*args)
    elif kind == "phi4":
        state["session"].forward_token(state["token"], state["position"])
    elif kind == "rwkv7":
        state["session"].forward_token(state["token"])
    else:
        state["owner"].plan.launch()
    return state["out"]


# ---- what a pass cannot do without -----------------------------------------------------------

def work(case):
    kind = case["kind"]
    size = lambda r, c: native.tensor_bytes(FORMATS[case["fmt"]], r, c)
    if kind == "matvec":
        r, c = case["rows"], case["cols"]
        return {"bytes": case["calls"] * (size(r, c) + 4 * r) + 4 * c, "flops": case["calls"] * 2 * r * c}
    if kind == "products":
        shapes = _shapes(case)
        return {"bytes": case["layers"] * sum(size(r, c) + 4 * (r + c) for r, c in shapes),
                "flops": case["layers"] * sum(2 * r * c for r, c in shapes)}
    if kind == "chain":
        h, f, q = case["hidden"], case["ffn"], case["qkv"]
        shapes = [(q, h), (h, h), (2 * f, h), (h, f)]
        return {"bytes": case["layers"] * (sum(size(r, c) for r, c in shapes) + 4 * (4 * h + q + f)),
                "flops": case["layers"] * sum(2 * r * c for r, c in shapes)}
    if kind == "prefill":
        shapes, m = _shapes(case), case["m"]
        return {"bytes": sum(size(r, c) + 4 * m * r for r, c in shapes) + 2 * m * sum({c for _, c in shapes}),
                "flops": sum(2 * m * r * c for r, c in shapes)}
    if kind == "batch":
        n, v, shapes = case["layers"], case["valid"], _layer_shapes(case)
        row = (2 if case["cache"] == "f16" else 4) * 128 * case["kv_heads"]
        seen = case["start"] + v
        return {"bytes": n * (sum(size(r, c) for r, c in shapes) + 2 * row * seen + 8 * case["hidden"]) +
                12 * v * case["hidden"],
                "flops": n * (2 * v * sum(r * c for r, c in shapes) + 4 * v * seen * 128 * case["heads"])}
    if kind == "attention":
        n, seen = case["layers"], case["position"] + 1
        return {"bytes": n * (4 * 128 * case["kv_heads"] * seen + 4 * 128 * (2 * case["heads"] + 2 * case["kv_heads"])),
                "flops": n * 4 * 128 * case["heads"] * seen}
    if kind == "gqa":
        n, d, seen = case["layers"], case["head"], case["position"] + 1
        e = 2 if case["cache"] == "f16" else 4
        return {"bytes": n * (2 * e * d * case["kv_heads"] * seen + 8 * d * case["heads"]),
                "flops": n * 4 * d * case["heads"] * seen}
    if kind == "phi4":
        cfg = _phi4_config(case)
        return {"bytes": cfg.weight_bytes_per_token() + cfg.kv_bytes(case["position"] + 1) + 4 * case["vocab"],
                "flops": 2 * (case["layers"] * sum(r * c for r, c in _layer_shapes(case)) + case["vocab"] * case["hidden"])
                + 4 * 128 * case["heads"] * (case["position"] + 1) * case["layers"]}
    cfg = _rwkv_config(case)
    macs = sum(r * c for l in range(case["layers"]) for r, c in cfg.matrix_shapes(l).values())
    return {"bytes": cfg.weight_bytes_per_token() + 4 * case["vocab"],
            "flops": 2 * (macs + case["vocab"] * cfg.hidden + 4 * case["layers"] * case["heads"] * 64 * 64)}


def tolerance(case):
    """About four times the distance to exact() that each kind shows."""
    return {
        "matvec": {"rel": 2.5e-6},                    # FP32 sums; x on a 21-bit grid per block in some forms
        "products": {"rel": 2.5e-6},
        "chain": {"rel": 2e-5},
        "prefill": {"rel": 7e-3},                     # weights rounded to bf16
        "batch": {"rel": 1e-4, "max": 4e-3},          # appended cache rows may round to the next fp16 value
        "attention": {"rel": 4e-4, "max": 4e-3},      # as above; FP32 angles of up to `position` radians
        "gqa": {"rel": 2.5e-6},
        "phi4": {"rel": 2e-4, "max": 4e-3},
        "rwkv7": {"rel": 1e-5},
    }[case["kind"]]


# ---- the same results in 64 bits ------------------------------------------------------------

def _dequant(fmt, w, rows, cols):
    if fmt in ("f16", "f32"):
        return w.view(torch.float16 if fmt == "f16" else torch.float32).reshape(rows, cols).to(F64)
    if fmt == "q8_0":
        b = w.reshape(-1, 34)
        d = b[:, :2].contiguous().view(torch.float16).to(F64)
        return (d * b[:, 2:].contiguous().view(torch.int8).to(F64)).reshape(rows, cols)
    if fmt == "q4_0":
        b = w.reshape(-1, 18)
        d = b[:, :2].contiguous().view(torch.float16).to(F64)
        return (d * (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).to(F64) - 8)).reshape(rows, cols)
    b = w.reshape(-1, 144)
    d, dmin = (b[:, i:i + 2].contiguous().view(torch.float16).to(F64).reshape(-1, 1, 1) for i in (0, 2))
    lo, mid, hi = b[:, 4:8], b[:, 8:12], b[:, 12:16]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1).to(F64).unsqueeze(2)
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1).to(F64).unsqueeze(2)
    q = b[:, 16:].reshape(-1, 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).to(F64)
    return (d * sc * q - dmin * mn).reshape(rows, cols)


def _mul(fmt, w, rows, cols, x):
    """x [..., cols] times the transposed weights, in row slices that bound the memory."""
    step, row = 32768, w.numel() // rows
    parts = [x @ _dequant(fmt, w[i * row:min(i + step, rows) * row], min(step, rows - i), cols).T
             for i in range(0, rows, step)]
    return torch.cat(parts, -1)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.to(F64)


def _silu_up(gu):
    g, u = gu.chunk(2, -1)
    return g / (1 + torch.exp(-g)) * u


def _rotate(v, positions, freq, rotary):
    """v [rows, heads, 128]; the FP32 angles the operators are defined on, rotated in 64 bits."""
    a = (positions.to(torch.float32)[:, None] * freq[None, :]).to(F64)[:, None, :]
    half = rotary // 2
    left, right = v[..., :half], v[..., half:rotary]
    return torch.cat([left * a.cos() - right * a.sin(), right * a.cos() + left * a.sin(), v[..., rotary:]], -1)


def _attend(q, k, v):
    """q [heads, d], k and v [kv_heads, positions, d]."""
    group = q.shape[0] // k.shape[0]
    q = q.reshape(k.shape[0], group, -1)
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])
    return torch.matmul(torch.softmax(s, -1), v.contiguous()).reshape(-1)


def _layernorm(x, w, b, eps=1e-5):
    c = x - x.mean(-1, keepdim=True)
    return c / torch.sqrt((c * c).mean(-1, keepdim=True) + eps) * w.to(F64) + b.to(F64)


def exact(case, seed):
    inp = _inputs(case, seed)
    kind, fmt = case["kind"], case.get("fmt")
    if kind == "matvec":
        return [_mul(fmt, w, case["rows"], case["cols"], inp["x"].to(F64)) for w in inp["w"]]
    if kind == "products":
        shapes = _shapes(case)
        return [_mul(fmt, w, r, c, inp["x"][c].to(F64)) for ws in inp["w"] for (r, c), w in zip(shapes, ws)]
    if kind == "chain":
        h, f, q = case["hidden"], case["ffn"], case["qkv"]
        x, out = inp["h"].to(F64), []
        for (wqkv, wo, wup, wdown), (n1, n2) in zip(inp["w"], inp["norms"]):
            qkv = _mul(fmt, wqkv, q, h, _rms(x, n1))
            h1 = x + _mul(fmt, wo, h, h, qkv[:h])
            act = _silu_up(_mul(fmt, wup, 2 * f, h, _rms(h1, n2)))
            x = h1 + _mul(fmt, wdown, h, f, act)
            out += [qkv, h1, act, x]
        return out
    if kind == "prefill":
        return [_mul(fmt, w, r, c, inp["x"][c].to(F64)) for (r, c), w in zip(_shapes(case), inp["w"])]
    if kind == "batch":
        return _exact_batch(case, inp)
    if kind == "attention":
        heads, kv, at = case["heads"], case["kv_heads"], case["position"]
        pos, freq, out = inp["position"], _frequencies(case["rotary"]), []
        for l in range(case["layers"]):
            rows = inp["qkv"][l].to(F64).reshape(1, -1, 128)
            q = _rotate(rows[:, :heads], pos, freq, case["rotary"])[0]
            inp["k"][l, :, at] = _rotate(rows[:, heads:heads + kv], pos, freq, case["rotary"])[0].half()
            inp["v"][l, :, at] = rows[0, heads + kv:].half()
            out.append(_attend(q, inp["k"][l, :, :at + 1].to(F64), inp["v"][l, :, :at + 1].to(F64)))
        return [torch.stack(out), inp["k"][:, :, at].to(F64), inp["v"][:, :, at].to(F64)]
    if kind == "gqa":
        kv, d, seen = case["kv_heads"], case["head"], case["position"] + 1
        rows = lambda t: t[:seen].to(F64).reshape(seen, kv, d).transpose(0, 1)
        return torch.stack([_attend(inp["q"][l].to(F64).reshape(-1, d), rows(inp["k"][l]), rows(inp["v"][l]))
                            for l in range(case["layers"])])
    if kind == "phi4":
        return _exact_phi4(case, inp)
    return _exact_rwkv7(case, inp)


def _exact_batch(case, inp):
    n, v, h, f, heads, kv = (case[k] for k in ("layers", "valid", "hidden", "ffn", "heads", "kv_heads"))
    fmt, start = case["fmt"], case["start"]
    pos = torch.arange(start, start + v, device="cuda")
    x = inp["h"][:v].to(F64)
    shapes = _layer_shapes(case)
    for l in range(n):
        mul = lambda i, a: _mul(fmt, inp["w"][l][i], *shapes[i], a)
        rows = mul(0, _rms(x, inp["norms"][l][0])).reshape(v, -1, 128)
        q = _rotate(rows[:, :heads], pos, inp["freq"], 96)
        inp["k"][l, start:start + v] = _rotate(rows[:, heads:heads + kv], pos, inp["freq"], 96).reshape(v, -1).to(inp["k"].dtype)
        inp["v"][l, start:start + v] = rows[:, heads + kv:].reshape(v, -1).to(inp["v"].dtype)
        cache = lambda t, s: t[l, :s].to(F64).reshape(s, kv, 128).transpose(0, 1)
        attn = torch.stack([_attend(q[r], cache(inp["k"], start + r + 1), cache(inp["v"], start + r + 1)) for r in range(v)])
        x = x + mul(1, attn)
        x = x + mul(3, _silu_up(mul(2, _rms(x, inp["norms"][l][1]))))
    whole = lambda t: torch.cat([t, torch.zeros(16 - v, h, device="cuda", dtype=F64)])
    return [whole(_rms(x, inp["out_norm"])), whole(x), inp["k"][:, start:start + v].to(F64),
            inp["v"][:, start:start + v].to(F64)]


def _exact_phi4(case, inp):
    h, heads, kv, at = case["hidden"], case["heads"], case["kv_heads"], case["position"]
    fmt, shapes = case["fmt"], _layer_shapes(case)
    pos, freq = torch.tensor([at], device="cuda"), _frequencies(96)
    row = inp["embed"].numel() // case["vocab"]
    x = _dequant("q8_0", inp["embed"][inp["token"] * row:(inp["token"] + 1) * row], 1, h)[0]
    for ws, (n1, n2), (k, v) in zip(inp["w"], inp["norms"], inp["kv"]):
        mul = lambda i, a: _mul(fmt, ws[i], *shapes[i], a)
        rows = mul(0, _rms(x, n1)).reshape(1, -1, 128)
        q = _rotate(rows[:, :heads], pos, freq, 96)[0]
        knew = _rotate(rows[:, heads:heads + kv], pos, freq, 96)[0].half()
        vnew = rows[0, heads + kv:].half()
        k, v = (torch.cat([c, new[:, None]], 1).to(F64) for c, new in ((k, knew), (v, vnew)))
        x = x + mul(1, _attend(q, k, v))
        x = x + mul(3, _silu_up(mul(2, _rms(x, n2))))
    return [_mul("q8_0", inp["head"], case["vocab"], h, _rms(x, inp["out_norm"])), knew.to(F64), vnew.to(F64)]


def _exact_rwkv7(case, inp):
    heads, fmt = case["heads"], case["fmt"]
    d = 64 * heads
    cfg = _rwkv_config(case)
    row = inp["embed"].numel() // case["vocab"]
    x = _layernorm(_dequant("q8_0", inp["embed"][inp["token"] * row:(inp["token"] + 1) * row], 1, d)[0], *inp["ln0"])
    v_first, prevs, states = None, [], []
    per_head = lambda t: t.reshape(heads, 64)
    for l, (L, (att_prev, ffn_prev, S)) in enumerate(zip(inp["layers"], inp["state"])):
        V = {k: L[k].to(F64) for k in ("w0", "a0", "v0", "k_k", "k_a", "r_k")}
        mul = lambda name, a: _mul(fmt, L[name], *cfg.matrix_shapes(1)[name], a)
        n = _layernorm(x, L["ln1_weight"], L["ln1_bias"])
        xr, xw, xk, xv, xa, xg = (n + (att_prev.to(F64) - n) * m for m in L["mix"].to(F64))
        r, k, v = mul("receptance", xr), mul("key", xk), mul("value", xv)
        decay = torch.exp(-0.606531 * torch.sigmoid(mul("w2", torch.tanh(mul("w1", xw))) + V["w0"]))
        a = torch.sigmoid(mul("a2", mul("a1", xa)) + V["a0"])
        gate = mul("g2", torch.sigmoid(mul("g1", xg)))
        kn = per_head(k * V["k_k"])
        kn = kn / torch.sqrt(torch.clamp((kn * kn).sum(-1, keepdim=True), min=1e-24))
        key = k + a * (k * V["k_a"]) - k * V["k_a"]
        if l == 0:
            value = v_first = v
        else:
            value = v + (v_first - v) * torch.sigmoid(mul("v2", mul("v1", xv)) + V["v0"])
        S = S.to(F64)
        S = S * per_head(decay)[:, None, :] + per_head(value)[:, :, None] * per_head(key)[:, None, :] - \
            (S * kn[:, None, :]).sum(-1, keepdim=True) * (kn * per_head(a))[:, None, :]
        y = (S * per_head(r)[:, None, :]).sum(-1)
        y = _layernorm(y, per_head(L["lnx_weight"]), per_head(L["lnx_bias"]), 64e-5)
        y = y + per_head(value) * (per_head(key) * per_head(r) * per_head(V["r_k"])).sum(-1, keepdim=True)
        x = x + mul("output", y.reshape(-1) * gate)
        prevs.append(n)
        states.append(S)
        n = _layernorm(x, L["ln2_weight"], L["ln2_bias"])
        x = x + mul("ffn_value", torch.relu(mul("ffn_key", n + (ffn_prev.to(F64) - n) * L["ffn_mix"].to(F64))) ** 2)
    return [_mul("q8_0", inp["head"], case["vocab"], d, _layernorm(x, *inp["ln_out"]))] + prevs + states
