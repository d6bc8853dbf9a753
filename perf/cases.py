"""The work that a user of this framework has it do, as measurable cases.

`listed()` names twelve of them and `draw()` gives more from the same ranges.
`prepare(case, seed)` makes what a program holds before the call (operands,
outputs, handles, workspaces, a captured graph), `run(state)` is one pass
through the public entry points, `exact(case, seed)` the same results in
64 bits from plain torch, without this package. `work(case)` counts what a
pass cannot do without and `tolerance(case)` how far another correct
implementation at the same precision may be.

Operands follow what the paths meet in a model: weights are normal and
quantized per block (the quantizers below are plain ones: block maxima, no
search), activations are normal with a few channels ten times larger.
"""
from __future__ import annotations

import functools

import torch

import vortx_amd as vx

DEV = "cuda:0"
QTYPE = {"q4_0": vx.VX_Q4_0, "q8_0": vx.VX_Q8_0, "q4_k": vx.VX_Q4_K}
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144)}  # weights, bytes


# ----------------------------------------------------------------- cases
def listed():
    return [
        # One matrix-vector product of a decode step, launched by itself: the
        # up projection at batch 1, where a call's latency is what counts.
        {"name": "decode_q4_0", "op": "gemv", "quant": "q4_0", "rows": 11008, "cols": 4096, "batch": 1, "x": "int8"},
        # A decode step's seven projections of one layer (grouped-query
        # attention and a gated MLP) captured in a graph, as a serving loop
        # replays them for each token.
        {"name": "decode_layer_q4_k", "op": "layer", "quant": "q4_k", "hidden": 4096, "kv": 1024, "inner": 14336,
         "batch": 1},
        # The down projection of eight sequences decoded together, with the
        # caller's workspace (three passes over K).
        {"name": "decode_batch_q4_0", "op": "gemv", "quant": "q4_0", "rows": 4096, "cols": 11008, "batch": 8,
         "x": "int8"},
        # Prefill: a projection over a prompt of 512 tokens.
        {"name": "prefill_q4_k", "op": "gemv", "quant": "q4_k", "rows": 14336, "cols": 4096, "batch": 512, "x": "int8"},
        # A short prompt, of a ragged length, with the activations kept in f32.
        {"name": "prefill_q8_0_f32x", "op": "gemv", "quant": "q8_0", "rows": 4096, "cols": 4096, "batch": 67,
         "x": "f32"},
        # The largest call: a dense projection in f32.
        {"name": "gemm_large", "op": "gemm", "n": 1, "M": 4096, "N": 11008, "K": 4096, "ta": False, "tb": False,
         "alpha": 1.0, "beta": 0.0},
        # A dense layer's training step: forward, the input's gradient (B
        # transposed) and the weight's gradient added to what is there (A
        # transposed, beta 1).
        {"name": "dense_train", "op": "dense", "tokens": 1000, "inp": 1024, "out": 4096},
        # Sizes that are multiples of nothing, B a transposed view, scaled.
        {"name": "gemm_ragged", "op": "gemm", "n": 1, "M": 1000, "N": 1111, "K": 777, "ta": False, "tb": True,
         "alpha": 0.5, "beta": 0.0},
        # A few rows through a dense layer whose weights are stored [N, K].
        {"name": "gemm_skinny", "op": "gemm", "n": 1, "M": 8, "N": 11008, "K": 4096, "ta": False, "tb": True,
         "alpha": 1.0, "beta": 0.0},
        # The smallest call.
        {"name": "gemm_tiny", "op": "gemm", "n": 1, "M": 24, "N": 20, "K": 64, "ta": False, "tb": False,
         "alpha": 1.0, "beta": 0.0},
        # f32 weights to blocks and back (what a converter does to write a
        # file and to report its error).
        {"name": "convert_q4_0", "op": "convert", "quant": "q4_0", "rows": 14336, "cols": 4096},
        # The keys of a batch laid out [batch, tokens, heads, dim] made
        # contiguous as [batch, heads, dim, tokens].
        {"name": "contiguous_keys", "op": "copy", "sizes": "2,1000,32,128", "order": "0,2,3,1"},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    op = rng.choice(["gemv", "gemv", "gemv", "layer", "gemm", "gemm", "gemm", "dense", "convert", "copy"])
    if op == "gemv":
        quant = rng.choice(["q4_0", "q8_0", "q4_k"])
        unit = 256 if quant == "q4_k" else 64
        c = {"op": op, "quant": quant, "rows": _log(rng, 256, 32000), "cols": unit * _log(rng, 1024 // unit, 16384 // unit)}
        kind = rng.choice(["one", "batch", "prefill", "f32"])
        if kind == "one":
            c.update(batch=1, x=rng.choice(["int8", "f32"]))
        elif kind == "batch":
            c.update(batch=rng.randint(2, 16), x="int8")
        elif kind == "prefill":
            c.update(batch=_log(rng, 17, 512), x="int8")
        else:
            c.update(batch=_log(rng, 2, 128), x="f32")
        while c["rows"] * c["cols"] * c["batch"] > 3e10:  # no more than the largest listed ones
            c["rows"] = c["rows"] // 2 + 1
        return c
    if op == "layer":
        quant = rng.choice(["q4_0", "q8_0", "q4_k"])
        hidden = 256 * rng.randint(4, 20)
        return {"op": op, "quant": quant, "hidden": hidden, "kv": 64 * rng.randint(4, hidden // 64),
                "inner": 256 * rng.randint(hidden // 128, hidden // 64), "batch": rng.choice([1, 1, 2, 4])}
    if op == "gemm":
        kind = rng.choice(["any", "any", "skinny", "heads", "tiny"])
        c = {"op": op, "n": 1, "M": _log(rng, 32, 4096), "N": _log(rng, 32, 8192), "K": _log(rng, 32, 8192),
             "ta": rng.random() < 0.25, "tb": rng.random() < 0.5, "alpha": rng.choice([1.0, 0.5]),
             "beta": rng.choice([0.0, 0.0, 1.0])}
        if rng.random() < 0.5:  # as most layers are sized
            for d in ("M", "N", "K"):
                c[d] = -(-c[d] // 32) * 32
        if kind == "skinny":
            c.update(M=rng.randint(1, 31), N=_log(rng, 1024, 16384), K=_log(rng, 1024, 8192), ta=False)
        elif kind == "heads":
            c.update(n=rng.randint(2, 64), M=_log(rng, 32, 1024), N=_log(rng, 32, 1024), K=rng.choice([64, 80, 128]), ta=False)
        elif kind == "tiny":
            c.update(M=rng.randint(1, 31), N=rng.randint(1, 31), K=_log(rng, 8, 512), ta=False)
        while c["M"] * c["N"] * c["K"] > 1.8e11:
            c["N"] = c["N"] // 2 + 1
        return c
    if op == "dense":
        return {"op": op, "tokens": _log(rng, 64, 2048), "inp": _log(rng, 256, 4096), "out": _log(rng, 256, 4096)}
    if op == "convert":
        quant = rng.choice(["q4_0", "q8_0", "q4_k"])
        unit = BLOCK[quant][0]
        return {"op": op, "quant": quant, "rows": _log(rng, 256, 14336), "cols": unit * _log(rng, 512 // unit, 4096 // unit)}
    sizes = [rng.randint(1, 4), _log(rng, 16, 2048), _log(rng, 2, 48), rng.choice([32, 64, 80, 100, 128])]
    return {"op": op, "sizes": ",".join(map(str, sizes)), "order": rng.choice(["0,2,1,3", "0,2,3,1", "0,3,1,2", "1,0,3,2"])}


# -------------------------------------------------------------- operands
def _normal(shape, seed, scale=1.0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * scale


def _activations(batch, cols, seed):
    """[batch, cols], one channel in 64 ten times larger."""
    x = _normal((batch, cols), seed)
    x[:, seed % 64::64] *= 10.0
    return x


def _f16_bytes(v):
    h = v.to(torch.float16).contiguous()
    return h.view(torch.uint8).reshape(*h.shape, 2)


def _blocks(quant, rows, cols, seed):
    """Normal weights [rows, cols] as uint8 blocks [rows, cols / QK * bytes]."""
    qk, nbytes = BLOCK[quant]
    w = _normal((rows, cols), seed, cols ** -0.5).reshape(rows, cols // qk, qk)
    if quant == "q8_0":
        d = (w.abs().amax(-1) / 127).half().float().clamp_min(1e-7)
        q = (w / d[..., None]).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([_f16_bytes(d), q], -1).reshape(rows, -1)
    if quant == "q4_0":
        d = (w.abs().amax(-1) / 7.5).half().float().clamp_min(1e-7)
        q = (w / d[..., None] + 8).round_().clamp_(0, 15).to(torch.uint8)
        return torch.cat([_f16_bytes(d), q[..., :16] | (q[..., 16:] << 4)], -1).reshape(rows, -1)
    w = w.reshape(rows, cols // 256, 8, 32)
    low = (-w.amin(-1)).clamp_min_(0)
    step = (w.amax(-1) + low) / 15
    d = (step.amax(-1) / 63).half().float().clamp_min(1e-7)
    dmin = (low.amax(-1) / 63).half().float().clamp_min(1e-7)
    sc = (step / d[..., None]).round_().clamp_(1, 63)
    m = (low / dmin[..., None]).round_().clamp_(0, 63)
    q = ((w + (dmin[..., None] * m)[..., None]) / (d[..., None] * sc)[..., None]).round_().clamp_(0, 15).to(torch.uint8)
    sc, m = sc.to(torch.uint8), m.to(torch.uint8)
    packed = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), m[..., :4] | ((m[..., 4:] >> 4) << 6),
                        (sc[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)], -1)
    q = q.reshape(rows, cols // 256, 4, 2, 32)
    nib = (q[..., 0, :] | (q[..., 1, :] << 4)).reshape(rows, cols // 256, 128)
    return torch.cat([_f16_bytes(d), _f16_bytes(dmin), packed, nib], -1).reshape(rows, -1)


def _decoded(quant, blocks, cols):
    """The blocks' values in 64 bits, [rows, cols]."""
    qk, nbytes = BLOCK[quant]
    b = blocks.reshape(blocks.shape[0], cols // qk, nbytes)
    half = lambda at: b[..., at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if quant == "q8_0":
        return (half(0) * b[..., 2:].contiguous().view(torch.int8).double()).reshape(-1, cols)
    if quant == "q4_0":
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).double() - 8
        return (half(0) * q).reshape(-1, cols)
    p = b[..., 4:16]
    sc = torch.cat([p[..., :4] & 63, (p[..., 8:] & 15) | ((p[..., :4] >> 6) << 4)], -1).double()
    m = torch.cat([p[..., 4:8] & 63, (p[..., 8:] >> 4) | ((p[..., 4:8] >> 6) << 4)], -1).double()
    nib = b[..., 16:].reshape(b.shape[0], -1, 4, 32)
    q = torch.stack([nib & 15, nib >> 4], -2).reshape(b.shape[0], -1, 8, 32).double()
    return ((half(0) * sc)[..., None] * q - (half(2) * m)[..., None]).reshape(-1, cols)


def _times(blocks, quant, cols, x):
    """x [batch, cols] times the decoded rows, [batch, rows] in 64 bits, some rows at a time."""
    x = x.double()
    return torch.cat([x @ _decoded(quant, part, cols).t() for part in blocks.split(4096)], 1)


@functools.lru_cache(maxsize=None)
def _gemv():
    return vx.QuantGemv(0)


@functools.lru_cache(maxsize=None)
def _gemm():
    return vx.Gemm(0)


@functools.lru_cache(maxsize=None)
def _contiguous():
    return vx.Contiguous(0)


def _layer_shapes(c):
    """(rows, cols) of the q, k, v, output, gate, up and down projections."""
    h, kv, inner = c["hidden"], c["kv"], c["inner"]
    return [(h, h), (kv, h), (kv, h), (h, h), (inner, h), (inner, h), (h, inner)]


def _matrix(c, seed, which):
    """An operand of a product as the program stores it: [n, rows, cols], rows and cols exchanged if it is used transposed."""
    r, k, t = (c["M"], c["K"], c["ta"]) if which == 0 else (c["K"], c["N"], c["tb"])
    shape = (k, r) if t else (r, k)
    return _normal((c["n"], *shape) if c["n"] > 1 else shape, seed * 4 + which, 1.0 if which == 0 else c["K"] ** -0.5)


def _view(t, transposed):
    return t.transpose(-1, -2) if transposed else t


def _start_of_out(c, seed):
    shape = (c["M"], c["N"])
    return _normal((c["n"], *shape) if c["n"] > 1 else shape, seed * 4 + 2)


def _dense_operands(c, seed):
    t, i, o = c["tokens"], c["inp"], c["out"]
    return (_normal((t, i), seed * 4), _normal((i, o), seed * 4 + 1, i ** -0.5), _normal((t, o), seed * 4 + 2, 0.01),
            _normal((i, o), seed * 4 + 3, 0.01))


def _ints(text):
    return [int(v) for v in text.split(",")]


# ------------------------------------------------------------------ cases
def prepare(case, seed):
    c, op = case, case["op"]
    s = {"op": op}
    if op == "gemv":
        s["w"] = vx.QWeight(_blocks(c["quant"], c["rows"], c["cols"], seed * 2), QTYPE[c["quant"]], c["rows"], c["cols"])
        x = _activations(c["batch"], c["cols"], seed * 2 + 1)
        s["y"] = torch.empty((c["batch"], c["rows"]), device=DEV)
        s["f32"] = c["x"] == "f32"
        s["ws"] = vx.QuantGemv.workspace(s["w"], c["batch"]) if c["batch"] > 1 and not s["f32"] else None
        # activations and results are stored [batch, features]; the views are [features, batch]
        s["xv"], s["yv"] = (x[0], s["y"][0]) if c["batch"] == 1 else (x.t(), s["y"].t())
        _gemv()
    elif op == "layer":
        w = [vx.QWeight(_blocks(c["quant"], r, k, seed * 16 + i), QTYPE[c["quant"]], r, k)
             for i, (r, k) in enumerate(_layer_shapes(c))]
        x = [_activations(c["batch"], k, seed * 16 + 8 + i) for i, k in enumerate((c["hidden"], c["hidden"], c["hidden"], c["inner"]))]
        x = [x[0], x[0], x[0], x[1], x[2], x[2], x[3]]
        y = [torch.empty((c["batch"], r), device=DEV) for r, _ in _layer_shapes(c)]
        ws = vx.QuantGemv.workspace(max(w, key=lambda v: v.cols), c["batch"])
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        gv = _gemv()
        torch.cuda.synchronize()
        with torch.cuda.stream(stream), torch.cuda.graph(graph, stream=stream):
            for wi, xi, yi in zip(w, x, y):
                gv.dispatch(yi.t(), wi, xi.t(), stream=stream, workspace=ws if c["batch"] > 1 else None)
        s.update(w=w, x=x, y=y, ws=ws, graph=graph)
    elif op == "gemm":
        a, b = _matrix(c, seed, 0), _matrix(c, seed, 1)
        s.update(a=_view(a, c["ta"]), b=_view(b, c["tb"]), out=_start_of_out(c, seed), alpha=c["alpha"], beta=c["beta"],
                 plain=c["alpha"] == 1.0 and c["beta"] == 0.0)
        _gemm()
    elif op == "dense":
        x, w, dy, dw = _dense_operands(c, seed)
        s.update(x=x, w=w, dy=dy, dw=dw, y=torch.empty_like(dy), dx=torch.empty_like(x))
        _gemm()
    elif op == "convert":
        qk, nbytes = BLOCK[c["quant"]]
        data = torch.empty((c["rows"], c["cols"] // qk * nbytes), dtype=torch.uint8, device=DEV)
        s.update(x=_normal((c["rows"], c["cols"]), seed, c["cols"] ** -0.5), data=data,
                 w=vx.QWeight(data, QTYPE[c["quant"]], c["rows"], c["cols"]),
                 back=torch.empty((c["rows"], c["cols"]), device=DEV))
        _gemv()
    else:
        view = _normal(_ints(c["sizes"]), seed).permute(_ints(c["order"]))
        s.update(view=view, out=torch.empty(tuple(view.shape), device=DEV))
        _contiguous()
    return s


def run(state):
    s, op = state, state["op"]
    if op == "gemv":
        _gemv().dispatch(s["yv"], s["w"], s["xv"], x_f32=s["f32"], workspace=s["ws"])
        return s["y"]
    if op == "layer":
        s["graph"].replay()
        return s["y"]
    if op == "gemm":
        if s["plain"]:
            _gemm().dispatch(s["out"], s["a"], s["b"])
        else:
            _gemm().dispatch_ex(s["out"], s["a"], s["b"], alpha=s["alpha"], beta=s["beta"])
        return s["out"]
    if op == "dense":
        g = _gemm()
        g.dispatch(s["y"], s["x"], s["w"])
        g.dispatch(s["dx"], s["dy"], s["w"].t())
        g.dispatch_ex(s["dw"], s["x"].t(), s["dy"], beta=1.0)
        return s["y"], s["dx"], s["dw"]
    if op == "convert":
        _gemv().quantize(s["w"], s["x"])
        _gemv().dequantize(s["back"], s["w"])
        return s["data"], s["back"]
    _contiguous().launch(s["out"], s["view"])
    return s["out"]


def exact(case, seed):
    c, op = case, case["op"]
    if op == "gemv":
        x = _activations(c["batch"], c["cols"], seed * 2 + 1)
        return _times(_blocks(c["quant"], c["rows"], c["cols"], seed * 2), c["quant"], c["cols"], x)
    if op == "layer":
        x = [_activations(c["batch"], k, seed * 16 + 8 + i) for i, k in enumerate((c["hidden"], c["hidden"], c["hidden"], c["inner"]))]
        x = [x[0], x[0], x[0], x[1], x[2], x[2], x[3]]
        return [_times(_blocks(c["quant"], r, k, seed * 16 + i), c["quant"], k, x[i])
                for i, (r, k) in enumerate(_layer_shapes(c))]
    if op == "gemm":
        a, b = (_view(_matrix(c, seed, i), t).double() for i, t in ((0, c["ta"]), (1, c["tb"])))
        out = c["alpha"] * (a @ b)
        return out + c["beta"] * _start_of_out(c, seed).double() if c["beta"] else out
    if op == "dense":
        x, w, dy, dw = (t.double() for t in _dense_operands(c, seed))
        return x @ w, dy @ w.t(), dw + x.t() @ dy
    if op == "copy":
        return _normal(_ints(c["sizes"]), seed).permute(_ints(c["order"])).contiguous().double()
    return None  # convert: bytes, and the values that they stand for


def _gemv_work(quant, rows, cols, batch):
    qk, nbytes = BLOCK[quant]
    return rows * (cols // qk) * nbytes + 4 * batch * (rows + cols), 2 * rows * cols * batch


def work(case):
    c, op = case, case["op"]
    if op == "gemv":
        nbytes, flops = _gemv_work(c["quant"], c["rows"], c["cols"], c["batch"])
    elif op == "layer":
        parts = [_gemv_work(c["quant"], r, k, c["batch"]) for r, k in _layer_shapes(c)]
        nbytes, flops = sum(p[0] for p in parts), sum(p[1] for p in parts)
    elif op == "gemm":
        m, n, k = c["M"], c["N"], c["K"]
        nbytes = 4 * c["n"] * (m * k + k * n + m * n * (2 if c["beta"] else 1))
        flops = 2 * c["n"] * m * n * k
    elif op == "dense":
        t, i, o = c["tokens"], c["inp"], c["out"]
        nbytes, flops = 4 * (2 * t * i + 2 * t * o + 3 * i * o), 6 * t * i * o
    elif op == "convert":
        qk, per = BLOCK[c["quant"]]
        n = c["rows"] * c["cols"]
        nbytes, flops = 8 * n + 2 * n // qk * per, 0
    else:
        n = 1
        for v in _ints(c["sizes"]):
            n *= v
        nbytes, flops = 8 * n, 0
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    op = case["op"]
    if op in ("convert", "copy"):
        return "exact"  # bytes, the values that they stand for, and moved bits
    if op == "layer" or (op == "gemv" and case["x"] == "int8"):
        # the activations carry 15 bits of their block's largest value: 3e-5 to 1e-4 off 64 bits
        return {"rel": 4e-4}
    return {"rel": 1e-5}  # sums in 32 bits: up to 2e-6 off 64 bits at K = 8192
