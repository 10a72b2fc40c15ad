"""The calls this framework is measured on.

Each case is one pass a user's program makes through the public entry
points: a decode step of a model's projections (cudalab_amd.decode), one or
several GEMVs (forward_into of an operator's extension object), or the
quantization of a weight matrix (quantize_w).  `listed()` names the cases,
`draw()` gives more of the same ranges: INT4, INT8, FP16 and FP32 weights,
matrices from under 1 MB to several hundred, row lengths from 256 to 65536,
aligned, odd and ragged sizes, eager calls and captured graphs.

Inputs come from the seed alone: W ~ N(0, 0.02) (decode: N(0, 1/K)) in fp16,
quantized symmetrically (INT4 per group of 128, INT8 per row), x ~ N(0, 1).
"""
import torch

GROUP = 128
VARIANT = {"int4gemv": "int4gemv_cdna4", "qgemv": "qgemv_cdna4",
           "gemv_f16": "gemv_cdna4", "gemv_f32": "gemv_cdna4"}
DTYPE = {"gemv_f16": torch.float16, "gemv_f32": torch.float32}
MOST_BYTES = 880_000_000        # of one pass (the 70B decode layers)


def _decode(name, op, mode, layers, hidden, inter, kv):
    return {"name": name, "kind": "decode", "op": op, "mode": mode, "layers": layers,
            "hidden": hidden, "inter": inter, "kv": kv}


def _gemv(name, op, mode, calls, n, k):
    return {"name": name, "kind": "gemv", "op": op, "mode": mode, "calls": calls,
            "n": n, "k": k}


def _quantize(name, op, n, k):
    return {"name": name, "kind": "quantize", "op": op, "n": n, "k": k}


def listed():
    return [
        # a draft model's two layers, called eagerly: five short launches a
        # layer, where the call and launch cost counts
        _decode("decode_small_int4_eager", "int4gemv", "grouped", 2, 1024, 2816, 256),
        # the main workload: a token through Llama-7B layers, weights in
        # INT4, replayed from a HIP graph
        _decode("decode_7b_int4_graph", "int4gemv", "graph", 4, 4096, 11008, 4096),
        # the same layers with INT8 weights, called eagerly
        _decode("decode_7b_int8_eager", "qgemv", "grouped", 4, 4096, 11008, 4096),
        # Llama-70B layers (grouped-query k/v, K-tiled down projection): the
        # largest pass
        _decode("decode_70b_int4_graph", "int4gemv", "graph", 2, 8192, 28672, 1024),
        # the headline shape, independent calls back to back over distinct
        # weights
        _gemv("int4_square_graph", "int4gemv", "graph", 16, 4096, 4096),
        # one rank's rows of a row-sharded 70B down projection: few, long rows
        _gemv("int4_short_long_graph", "int4gemv", "graph", 8, 1024, 28672),
        # a whole 70B down projection in INT8, one eager call
        _gemv("int8_down_70b", "qgemv", "eager", 1, 8192, 28672),
        # rows and columns of no round size (any K is in INT8's contract)
        _gemv("int8_ragged", "qgemv", "eager", 1, 4001, 4099),
        # a vocabulary head left in FP16
        _gemv("fp16_head", "gemv_f16", "eager", 1, 32000, 4096),
        # FP32 weights, the bench matrix's long-row shape
        _gemv("fp32_down", "gemv_f32", "eager", 1, 4096, 11008),
        # loading a model: the MLP projections' weights quantized on the device
        _quantize("quantize_int4_down", "int4gemv", 4096, 11008),
        _quantize("quantize_int8_up", "qgemv", 11008, 4096),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["decode", "gemv", "gemv", "gemv", "quantize"])
    if kind == "decode":
        op = rng.choice(["int4gemv", "qgemv"])
        kv = GROUP * _log(rng, 1, 16)
        hidden = kv * rng.choice([1, 2, 4, 8])
        hidden = hidden if hidden <= 8192 else kv
        inter = GROUP * max(1, round(hidden * rng.uniform(2.5, 3.6) / GROUP))
        per = sum(_wbytes(op, n, k) for n, k in _projections(hidden, inter, kv))
        layers = max(1, min(_log(rng, 1, 8), int(MOST_BYTES // per)))
        mode = rng.choice(["sequential", "grouped", "graph"])
        return {"kind": kind, "op": op, "mode": mode, "layers": layers,
                "hidden": hidden, "inter": inter, "kv": kv}
    if kind == "quantize":
        op = rng.choice(["int4gemv", "qgemv"])
        n, k = _log(rng, 256, 28672), _log(rng, 256, 28672)
        if op == "int4gemv" or rng.random() < 0.7:
            k = GROUP * max(1, k // GROUP)
        n = min(n, MOST_BYTES // (4 * k))
        return {"kind": kind, "op": op, "n": n, "k": k}
    op = rng.choice(["int4gemv", "int4gemv", "qgemv", "gemv_f16", "gemv_f32"])
    n, k = _log(rng, 256, 32768), _log(rng, 256, 65536)
    if op == "int4gemv":
        k = GROUP * max(1, k // GROUP)
    elif rng.random() < 0.7:
        k = 16 * max(1, k // 16)
    n = max(1, min(n, MOST_BYTES // (4 * k)))
    # enough calls that a pass is a piece of work and not one launch
    calls = max(1, min(16, 24_000_000 // _wbytes(op, n, k)))
    return {"kind": kind, "op": op, "mode": rng.choice(["eager", "graph"]),
            "calls": calls if calls > 1 else rng.choice([1, 2]), "n": n, "k": k}


# ------------------------------------------------------------------ inputs

def _projections(hidden, inter, kv):
    return ((hidden, hidden), (kv, hidden), (kv, hidden), (hidden, hidden),
            (inter, hidden), (inter, hidden), (hidden, inter))


def _wbytes(op, n, k):
    if op == "int4gemv":
        return n * k // 2 + n * (k // GROUP) * 2
    if op == "qgemv":
        return n * k + 4 * n
    return n * k * (2 if op == "gemv_f16" else 4)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _quantized(op, W):
    """The weight format, in plain torch: (q, scale), q int8 (N, K).  The
    scale is fp32 amax * fl(1/qmax), the quotient rounds half to even."""
    qmax = 7 if op == "int4gemv" else 127
    inv = (torch.ones((), dtype=torch.float32) / qmax).item()
    n, k = W.shape
    wf = W.float().reshape(n, -1, GROUP if op == "int4gemv" else k)
    s = wf.abs().amax(dim=2, keepdim=True) * inv
    q = torch.round(wf / torch.where(s == 0, torch.ones_like(s), s))
    q = q.clamp_(-qmax, qmax).masked_fill_(s == 0, 0.0).to(torch.int8).reshape(n, k)
    s = s.squeeze(2)
    return q, (s.half() if op == "int4gemv" else s.squeeze(1)).contiguous()


def _packed(q):
    u = (q & 15).to(torch.uint8)
    return (u[:, 0::2] | (u[:, 1::2] << 4)).contiguous()


def _gemv_set(case, g):
    """(W, scale, x) of one GEMV; scale is None for FP16 / FP32; an INT4 W
    comes unpacked (int8 values)."""
    op, n, k = case["op"], case["n"], case["k"]
    W = torch.randn(n, k, generator=g, device="cuda") * 0.02
    x = torch.randn(k, generator=g, device="cuda")
    if op in DTYPE:
        return W.to(DTYPE[op]), None, x.to(DTYPE[op])
    q, s = _quantized(op, W.half())
    return q, s, x.half()


def _decode_weights(case, seed):
    """The weights DecodeModel draws for this seed, layer by layer, and its
    input: what its constructor documents, in plain torch."""
    g = _generator(seed)
    layers = []
    for _ in range(case["layers"]):
        ws = []
        for n, k in _projections(case["hidden"], case["inter"], case["kv"]):
            W = (torch.randn(n, k, generator=g, device="cuda") / k ** 0.5).half()
            ws.append(_quantized(case["op"], W))
        layers.append(ws)
    return layers, torch.randn(case["hidden"], generator=g, device="cuda").half()


# --------------------------------------------------------------- the cases

def prepare(case, seed):
    if case["kind"] == "decode":
        from cudalab_amd.decode import DecodeModel
        m = DecodeModel(case["op"], case["layers"], seed=int(seed), hidden=case["hidden"],
                        inter=case["inter"], kv=case["kv"])
        step = {"grouped": m.step_grouped, "sequential": m.step_sequential}.get(case["mode"])
        if step is None:
            step = m.capture().replay
        outs = [L.out[name] for L in m.layers for name, _, _ in m.proj]
        return {"step": step, "outs": outs, "model": m}
    g = _generator(seed)
    if case["kind"] == "quantize":
        W = (torch.randn(case["n"], case["k"], generator=g, device="cuda") * 0.02).half()
        return {"quantize": _quantizer(case["op"]), "W": W}
    from cudalab_amd.build import build
    op = case["op"]
    ext = build("gemv" if op in DTYPE else op)
    calls = []
    for _ in range(case["calls"]):
        W, s, x = _gemv_set(case, g)
        W = _packed(W) if op == "int4gemv" else W
        out = torch.empty(case["n"], dtype=x.dtype, device="cuda")
        calls.append((W, x, out) if s is None else (W, s, x, out))
    variant = VARIANT[op]

    def step():
        for c in calls:
            ext.forward_into(variant, *c)

    outs = [c[-1] for c in calls]
    if case["mode"] == "eager":
        return {"step": step, "outs": outs}
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        step()
    torch.cuda.synchronize()
    return {"step": graph.replay, "outs": outs, "calls": calls}


def _quantizer(op):
    if op == "int4gemv":
        from cudalab_amd.int4gemv_quantize import quantize_w
    else:
        from cudalab_amd.qgemv_quantize import quantize_w
    return quantize_w


def run(state):
    if "quantize" in state:
        return state["quantize"](state["W"])
    state["step"]()
    return state["outs"]


def work(case):
    op = case["op"]
    if case["kind"] == "decode":
        shapes = _projections(case["hidden"], case["inter"], case["kv"])
        act = 2
        times = case["layers"]
    elif case["kind"] == "quantize":
        n, k = case["n"], case["k"]
        return {"bytes": 2 * n * k + _wbytes(op, n, k), "flops": 4 * n * k}
    else:
        shapes = ((case["n"], case["k"]),)
        act = 4 if op == "gemv_f32" else 2
        times = case["calls"]
    return {"bytes": times * sum(_wbytes(op, n, k) + act * (n + k) for n, k in shapes),
            "flops": times * sum(2 * n * k for n, k in shapes)}


def tolerance(case):
    """Measured against `exact`, about four times what is seen: one fp16
    rounding of each output (2.1e-4 of its norm), over the layers of a
    decode step where a flipped rounding travels on; fp32 sums."""
    if case["kind"] == "quantize":
        return "exact"
    if case["kind"] == "decode":
        return {"rel": 2.5e-3}
    return {"rel": 3e-6} if case["op"] == "gemv_f32" else {"rel": 8e-4}


def _product(op, W, s, x):
    """W x in 64 bits, in pieces of rows."""
    xd, out = x.double(), []
    rows = max(1, (1 << 26) // W.shape[1])
    for i in range(0, W.shape[0], rows):
        w = W[i:i + rows].double()
        if op == "int4gemv":
            w = (w.reshape(w.shape[0], -1, GROUP) * s[i:i + rows].double().unsqueeze(2)).flatten(1)
        y = torch.mv(w, xd)
        out.append(y * s[i:i + rows].double() if op == "qgemv" else y)
    return torch.cat(out)


def exact(case, seed):
    op = case["op"]
    if case["kind"] == "decode":
        layers, x = _decode_weights(case, seed)
        outs, rep = [], case["hidden"] // case["kv"]
        for (q, k, v, o, gate, up, down) in layers:
            # each projection in 64 bits on its fp16 input; what a projection
            # hands on is fp16, as the output buffers are
            y = [_product(op, *w, x) for w in (q, k, v)]
            heads = y[2].half().view(-1, 1, 128).expand(-1, rep, 128).reshape(-1)
            y.append(_product(op, *o, heads))
            y += [_product(op, *w, y[3].half()) for w in (gate, up)]
            y.append(_product(op, *down, y[5].half()))
            x = y[6].half()
            outs += y
        return outs
    g = _generator(seed)
    if case["kind"] == "quantize":
        # the format's own arithmetic: its bytes are the result
        W = (torch.randn(case["n"], case["k"], generator=g, device="cuda") * 0.02).half()
        q, s = _quantized(op, W)
        return (_packed(q) if op == "int4gemv" else q), s
    return [_product(op, *_gemv_set(case, g)) for _ in range(case["calls"])]
