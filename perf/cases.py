"""The work a serving program gives this library, as cases that can be timed.

A program that serves a GGUF model calls the library for the projections of
its decoder layers, between an attention of its own:

  attn  RMSNorm + Q8_1 of the residual, Q/K/V; Q8_1 of the attention's output
        (an input here), O added into the fp32 residual
  mlp   RMSNorm + Q8_1 of the residual, gate and up, SiLU(gate) * up + Q8_1,
        down added into the fp32 residual
  layer attn, then mlp on the residual it leaves
  head  the LM head's logits from the Q8_1 activations of the last norm

for M rows at a time: 1 when one sequence decodes, up to 32 when a batch
does, more when a batch is large or a prompt is read.  Each goes through the
entry points that serve the shape (the fused ones at small M).  Decode passes
(M <= 32) are captured once into a HIP graph and replayed, as the serving loop
replays its step, except where "graph" is False: a program that calls the
entry points one by one.  `layers` layers follow one another, each with
weights of its own.

Case values:
  kind, M, layers, graph
  hidden, q, kv, ffn, vocab   sizes (attn: q + 2 kv rows; head: vocab rows)
  quant    "q4_k_m" (Q4_K, down and head Q6_K) or "q8_0" (all Q8_0)
  layout   "raw" (GGUF rows), "row" (raw, but Q6_K / Q8_0 down and head as row-split
           copies: M <= 2) or "tiled" (load-time tiled copies: M <= 32)
  out      "f32" or "f16": what Q/K/V, gate, up and the logits are written as
  ws       True: a caller workspace and the ordered reductions (the same bits
           on every call); False: the plain entries, which may add with atomics

Sizes are the configurations of inferflux_amd/workloads.py (3B: hidden 2048,
Q/K/V 2048/256/256, FFN 11008; 14B: 5120, 5120/1024/1024, 13824; 32B: FFN
27648; vocabulary 151936) and, where drawn, others of the same kind.
"""
import torch

from inferflux_amd import ops

B3 = dict(hidden=2048, q=2048, kv=256, ffn=11008, vocab=151936)
B14 = dict(hidden=5120, q=5120, kv=1024, ffn=13824, vocab=151936)
B32 = dict(hidden=5120, q=5120, kv=1024, ffn=27648, vocab=151936)
EPS = 1e-6


def _case(name, kind, M, model, layers=1, graph=True, quant="q4_k_m", layout="raw", out="f32",
          ws=False):
    c = dict(kind=kind, M=M, layers=layers, graph=bool(graph and M <= 32), quant=quant,
             layout=layout, out=out, ws=ws, **model)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one sequence's attention projections by direct calls: the smallest
        # work, where launches and the host count
        _case("attn 3B M=1 direct", "attn", 1, B3, graph=False),
        # the decode step of a single sequence (chat): four layers, captured
        _case("layers 3B M=1", "layer", 1, B3, layers=4, layout="row"),
        # a few concurrent sequences, weights as the GGUF file has them
        _case("layers 3B M=6 raw", "layer", 6, B3, layers=3),
        # the same with the load-time tiled copies, an odd batch
        _case("layers 14B M=13 tiled", "layer", 13, B14, layers=1, layout="tiled"),
        # a full decode batch on the larger model
        _case("layers 14B M=32 tiled", "layer", 32, B14, layers=1, layout="tiled", ws=True),
        # the LM head of a decode batch: the widest single projection
        _case("head 3B M=8 Q6_K", "head", 8, B3),
        # a decode batch past 32, or a very short prompt
        _case("mlp 3B M=60", "mlp", 60, B3),
        # a short prompt, ragged, in a small model
        _case("layer 3B M=173", "layer", 173, B3, out="f16"),
        # a prefill chunk of 512 in a small model
        _case("layer 3B M=512", "layer", 512, B3),
        # the same in an 8-bit model
        _case("mlp 3B M=384 Q8_0", "mlp", 384, B3, quant="q8_0", out="f16"),
        # the 32B FFN on a prefill chunk, with the caller's workspace
        _case("mlp 32B M=512 ws", "mlp", 512, B32, ws=True),
        # a long prompt read at once, ragged
        _case("layer 14B M=1999", "layer", 1999, B14, out="f16", ws=True),
    ]


def draw(rng):
    """One more case: M over its whole range, sizes of models between 1B and
    32B, cut down where the work would pass the largest listed case's."""
    most = max(work(c)["flops"] for c in listed())
    while True:
        kind = rng.choice(["attn", "mlp", "layer", "layer", "head", "mlp"])
        M = int(round(2 ** rng.uniform(0, 11)))
        pick = rng.random()
        if pick < 0.4:
            model = dict(rng.choice([B3, B14, B32]))
        else:
            hidden = 256 * rng.randint(6, 24)
            model = dict(hidden=hidden, q=hidden, kv=hidden // rng.choice([1, 2, 4, 8]),
                         ffn=256 * int(hidden * rng.uniform(2.5, 5.5) / 256),
                         vocab=rng.choice([32000, 32003, 49152, 128256, 151936]))
        quant = rng.choice(["q4_k_m", "q4_k_m", "q8_0"])
        layout = "raw"
        if M <= 2 and rng.random() < 0.5:
            layout = "row"
        elif 3 <= M <= 32 and rng.random() < 0.5:
            layout = "tiled"
        c = _case(None, kind, M, model, layers=1 if kind == "head" or M > 8 else rng.randint(1, 3),
                  graph=rng.random() < 0.7, quant=quant, layout=layout,
                  out=rng.choice(["f32", "f16"]), ws=rng.random() < 0.5)
        if kind == "head" and M > 32:  # a prompt needs the logits of its last row
            continue
        if layout == "tiled" and c["out"] == "f16":  # fp16 splits need the workspace
            c["ws"] = True
        if work(c)["flops"] <= most:
            return c


# ------------------------------------------------------------------- inputs
def _types(c):
    """Quant types of (q/k/v/o/gate/up, down/head)."""
    return (ops.Q8_0, ops.Q8_0) if c["quant"] == "q8_0" else (ops.Q4_K, ops.Q6_K)


def _f16_bytes(n, lo, hi, g):
    d = torch.empty(n, device="cuda").uniform_(lo, hi, generator=g).half()
    return d.view(torch.uint8).view(n, 2)


def _blocks(qtype, n_rows, K, g):
    """Raw GGUF blocks of weights of about N(0, 0.04^2): random codes and
    sub-block scales, block scales within a factor of two."""
    n = n_rows * (K // ops.BLOCK_ELEMS[qtype])
    size = ops.BLOCK_BYTES[qtype]
    b = torch.randint(0, 256, (n, size), dtype=torch.uint8, device="cuda", generator=g)
    if qtype == ops.Q4_K:
        b[:, 0:2] = _f16_bytes(n, 1e-4, 2e-4, g)
        b[:, 2:4] = _f16_bytes(n, 7.5e-4, 1.5e-3, g)  # dmin: centres the values
    elif qtype == ops.Q6_K:
        b[:, 208:210] = _f16_bytes(n, 3e-5, 7e-5, g)
    else:
        b[:, 0:2] = _f16_bytes(n, 4e-4, 8e-4, g)
    return b.view(-1)


def _projections(c):
    """{name: (quant type, rows, K)} of one layer of the case."""
    t, td = _types(c)
    h, q, kv, f = c["hidden"], c["q"], c["kv"], c["ffn"]
    p = {}
    if c["kind"] == "head":
        return {"head": (td, c["vocab"], h)}
    if c["kind"] in ("attn", "layer"):
        p.update(q=(t, q, h), k=(t, kv, h), v=(t, kv, h), o=(t, h, q))
    if c["kind"] in ("mlp", "layer"):
        p.update(gate=(t, f, h), up=(t, f, h), down=(td, h, f))
    return p


def _draw_inputs(c, seed):
    """Weights per layer, norm weights, residual and attention outputs, from
    the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 2654435761 % (1 << 31) + 12345)
    M, h = c["M"], c["hidden"]

    def normal(rows, cols):
        return torch.randn(rows, cols, device="cuda", generator=g)

    x = normal(M, h)
    far = torch.randperm(h, device="cuda", generator=g)[:max(1, h // 100)]
    x[:, far] *= 20.0  # the outlier channels of a residual stream
    layers = []
    for _ in range(c["layers"]):
        w = {n: (t, rows, K, _blocks(t, rows, K, g)) for n, (t, rows, K) in _projections(c).items()}
        norms = [(1.0 + 0.1 * normal(1, h)[0]).half() for _ in range(2)]
        att = normal(M, c["q"]) * 0.5
        layers.append((w, norms, att))
    return x, layers


def _workspace(nbytes):
    return torch.zeros(max(int(nbytes), 256), dtype=torch.uint8, device="cuda")


class _State:
    """What the program keeps: weights in their layout, outputs, workspaces,
    and for a captured pass its graph."""


def _layer_state(c, w, norms, att):
    s = _State()
    M, od = c["M"], torch.float16 if c["out"] == "f16" else torch.float32
    small = torch.uint8
    h, f = c["hidden"], c["ffn"]
    s.w, s.att = {}, att
    s.norms = norms
    for n, (t, rows, K, raw) in w.items():
        if c["layout"] == "tiled":
            s.w[n] = ops.repack_tiled(t, raw, rows, K)
        elif c["layout"] == "row" and n in ("down", "head") and t in (ops.Q6_K, ops.Q8_0):
            s.w[n] = ops.repack(t, raw, rows, K)
        else:
            s.w[n] = (t, raw)

    def new(cols, dtype=od):
        return torch.empty(M, cols, dtype=dtype, device="cuda")

    s.a_hidden = new(h // 32 * 36, small)
    s.ws = {}
    if "q" in w:
        s.qkv = [new(w[n][1]) for n in "qkv"]
        s.a_att = new(c["q"] // 32 * 36, small)
        t = s.w["q"][0]
        if c["ws"] and M <= 32:
            s.ws["qkv"] = _workspace(ops.qgemv_workspace_bytes(t, [w[n][1] for n in "qkv"], M, h, od))
    if "gate" in w:
        s.a_ffn = new(f // 32 * 36, small)
        if M > 32:
            s.gate_up = [new(f), new(f)]
        else:
            need = ops.gate_up_silu_workspace_bytes(s.w["gate"][0], M, f, h)
            s.ws["gate_up"] = _workspace(need) if need else None
    if "head" in w:
        s.logits = new(c["vocab"])
        if c["ws"]:
            s.ws["head"] = _workspace(ops.qgemv_workspace_bytes(s.w["head"][0], [c["vocab"]], M, h, od))
    for n in ("o", "down"):
        if c["ws"] and n in w:
            t, rows, K = s.w[n][0], w[n][1], w[n][2]
            s.ws[n] = _workspace(ops.qgemv_workspace_bytes(t, [rows], M, K) if M <= 32 else
                                 ops.prefill_ordered_workspace_bytes(t, M, rows, K))
    if c["ws"] and M > 32:
        for n in ("q", "k", "v", "gate", "up"):
            if n in w:
                s.ws[n] = _workspace(ops.prefill_ordered_workspace_bytes(w[n][0], M, w[n][1], h, od))
    return s


def prepare(case, seed):
    x, layers = _draw_inputs(case, seed)
    s = _State()
    s.case, s.x, s.y = case, x, torch.empty_like(x)
    s.layers = [_layer_state(case, *l) for l in layers]
    if case["kind"] == "head":  # the last norm's activations, made by the step before
        L = s.layers[0]
        ops.rmsnorm_quantize_q8_1(x, L.norms[0], EPS, out=L.a_hidden)
    s.graph = None
    if case["graph"]:
        _forward(s)
        torch.cuda.synchronize()
        s.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s.graph):
            _forward(s)
        torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------- pass
def _group(c, s, names, outs, K, ws_name):
    """Sibling projections of the Q8_1 activations s.a_hidden."""
    M = c["M"]
    if M > 32 and c["ws"]:
        for n, y in zip(names, outs):
            t, W = s.w[n]
            ops.qgemm_prefill_ordered(t, W, s.a_hidden, M, y.shape[1], K, s.ws[n], out=y)
        return
    t = s.w[names[0]][0]
    ops.qgemv_grouped(t, [s.w[n][1] for n in names], s.a_hidden, M, [y.shape[1] for y in outs], K,
                      outs=outs, workspace=s.ws.get(ws_name))


def _add(c, s, name, A, y, K):
    """y += W . a, into the fp32 residual."""
    t, W = s.w[name]
    M, N = y.shape
    if M > 32 and c["ws"]:
        ops.qgemm_prefill_ordered(t, W, A, M, N, K, s.ws[name], out=y, mode=ops.ACCUM)
    else:
        ops.qgemv(t, W, A, M, N, K, out=y, mode=ops.ACCUM, workspace=s.ws.get(name))


def _attn(c, s, y):
    M, h, q = c["M"], c["hidden"], c["q"]
    fused = M <= 2 and s.w["q"][0] == ops.Q4_K
    rows = [o.shape[1] for o in s.qkv]
    if fused:
        ops.qgemv_grouped_rmsnorm(ops.Q4_K, [s.w[n][1] for n in "qkv"], y, s.norms[0], M, rows, h,
                                  EPS, outs=s.qkv)
        ops.qgemv_grouped_rmsnorm(ops.Q4_K, [s.w["o"][1]], s.att, None, M, [h], q, EPS, outs=[y],
                                  mode=ops.ACCUM)
        return
    ops.rmsnorm_quantize_q8_1(y, s.norms[0], EPS, out=s.a_hidden)
    _group(c, s, ["q", "k", "v"], s.qkv, h, "qkv")
    ops.quantize_q8_1(s.att, out=s.a_att)
    _add(c, s, "o", s.a_att, y, q)


def _mlp(c, s, y):
    M, h, f = c["M"], c["hidden"], c["ffn"]
    t, Wg = s.w["gate"]
    Wu = s.w["up"][1]
    if M <= 2 and t == ops.Q4_K and h <= 2048:
        ops.qgemv_gate_up_silu_rmsnorm(t, Wg, Wu, y, s.norms[1], M, f, h, EPS, q8_1_out=s.a_ffn,
                                       want_h=False)
    else:
        ops.rmsnorm_quantize_q8_1(y, s.norms[1], EPS, out=s.a_hidden)
        if M <= 32:
            ops.qgemv_gate_up_silu(t, Wg, Wu, s.a_hidden, M, f, h, q8_1_out=s.a_ffn, want_h=False,
                                   workspace=s.ws["gate_up"])
        else:
            _group(c, s, ["gate", "up"], s.gate_up, h, "gate_up")
            ops.silu_mul_quantize_q8_1(s.gate_up[0], s.gate_up[1], out=s.a_ffn)
    _add(c, s, "down", s.a_ffn, y, f)


def _forward(s):
    c = s.case
    if c["kind"] == "head":
        L = s.layers[0]
        t, W = L.w["head"]
        ops.qgemv(t, W, L.a_hidden, c["M"], c["vocab"], c["hidden"], out=L.logits,
                  workspace=L.ws.get("head"))
        return
    s.y.copy_(s.x)  # the embeddings, or the residual the layers before leave
    for L in s.layers:
        if c["kind"] != "mlp":
            _attn(c, L, s.y)
        if c["kind"] != "attn":
            _mlp(c, L, s.y)


def run(state):
    s = state
    if s.graph is not None:
        s.graph.replay()
    else:
        _forward(s)
    if s.case["kind"] == "head":
        return {"logits": s.layers[0].logits}
    got = {"residual": s.y}
    if s.case["kind"] != "mlp":
        got["qkv"] = [L.qkv for L in s.layers]
    if s.case["kind"] != "attn" and s.case["M"] > 32:
        got["gate_up"] = [L.gate_up for L in s.layers]
    return got


# ------------------------------------------------------------ what it takes
def work(case):
    c = case
    M, item = c["M"], 2 if c["out"] == "f16" else 4
    weights = values = 0
    for t, rows, K in _projections(c).values():
        weights += ops.weight_bytes(t, rows, K)
        values += rows * K
    L = c["layers"]
    if c["kind"] == "head":
        moved = M * (c["hidden"] // 32 * 36 + c["vocab"] * item)
    else:
        moved = 2 * M * c["hidden"] * 4  # residual in and out
        if c["kind"] != "mlp":
            moved += L * M * (c["q"] * 4 + (c["q"] + 2 * c["kv"]) * item)
        moved += L * 2 * c["hidden"] * 2  # norm weights
    return {"bytes": L * weights + moved, "flops": 2.0 * M * values * L}


def tolerance(case):
    """Sums in fp32 of 8-bit activations times 4- to 8-bit weights, compared with
    exact() and stated about four times wider.  Up to M = 16 a block's dot
    product is a whole number and the rest is fp32, but for the Q4_K minimum,
    which multiplies a block sum that Q8_1 keeps in fp16 (logits 7e-8 off, Q/K/V
    2e-4); above, weights and activations are rounded to fp16 (4.9e-4).  Where
    a result is quantized to Q8_1 again, as the next norm's or SiLU's output,
    such a difference moves some values across a rounding step of 1/254 of
    their block's largest: 3e-3 after an mlp, 7e-3 after a layer, 1.4e-2 after
    the second layer."""
    c = case
    if c["kind"] == "head":
        whole = c["M"] <= 16 and c["out"] == "f32"
        return {"rel": 1e-6 if whole else 2e-3}
    if c["kind"] == "attn" and c["layers"] == 1:
        return {"rel": 2e-3}
    if c["kind"] == "mlp" and c["layers"] == 1:
        return {"rel": 1.2e-2}
    return {"rel": 2.5e-2 if c["layers"] == 1 else 3e-2}


# ------------------------------------------------------------ in 64 bits
def _weights64(qtype, rows, K, raw):
    b = raw.view(-1, ops.BLOCK_BYTES[qtype])
    n = b.shape[0]

    def half(lo):
        return b[:, lo:lo + 2].contiguous().view(torch.float16).double()

    if qtype == ops.Q8_0:
        w = half(0) * b[:, 2:34].contiguous().view(torch.int8).double()
    elif qtype == ops.Q4_K:
        s = b[:, 4:16].short()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, 16:144].view(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(n, 8, 32).double()
        w = (half(0) * sc).unsqueeze(2) * q - (half(2) * mn).unsqueeze(2)
    else:
        ql = b[:, 0:128].view(n, 2, 1, 2, 32)
        qh = b[:, 128:192].view(n, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2).view(n, 2, 4, 32).short()
        high = torch.cat([(qh >> (2 * i)) & 3 for i in range(4)], 2).short()
        q = (low | (high << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(n, 2, 4, 2, 1)
        w = half(208).view(n, 1, 1, 1, 1) * sc * q.view(n, 2, 4, 2, 16).double()
    return w.reshape(rows, K)


def _q8_64(x):
    """The values of x's Q8_1 blocks."""
    M, K = x.shape
    b = x.view(M, K // 32, 32)
    amax = b.abs().amax(2, keepdim=True)
    inv = torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))
    return ((amax / 127.0).half().double() * torch.round(b * inv)).view(M, K)


def _times64(w, a):
    t, rows, K, raw = w
    per = ops.weight_bytes(t, 1, K)
    step = max(1, (1 << 27) // K)
    parts = [a @ _weights64(t, min(step, rows - r), K, raw[r * per:(r + min(step, rows - r)) * per]).t()
             for r in range(0, rows, step)]
    return torch.cat(parts, 1)


def exact(case, seed):
    x, layers = _draw_inputs(case, seed)
    x = x.double()

    def norm(v, w):
        return _q8_64(v / torch.sqrt((v * v).mean(1, keepdim=True) + EPS) * w.double())

    if case["kind"] == "head":
        w, norms, _ = layers[0]
        return {"logits": _times64(w["head"], norm(x, norms[0]))}
    got = {"qkv": [], "gate_up": []}
    for w, norms, att in layers:
        if case["kind"] != "mlp":
            a = norm(x, norms[0])
            got["qkv"].append([_times64(w[n], a) for n in "qkv"])
            x = x + _times64(w["o"], _q8_64(att.double()))
        if case["kind"] != "attn":
            a = norm(x, norms[1])
            g, u = _times64(w["gate"], a), _times64(w["up"], a)
            got["gate_up"].append([g, u])
            x = x + _times64(w["down"], _q8_64(torch.nn.functional.silu(g) * u))
    got["residual"] = x
    if case["kind"] == "mlp":
        del got["qkv"]
    if case["kind"] == "attn" or case["M"] <= 32:
        del got["gate_up"]
    return got
