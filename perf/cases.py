"""What a program that serves an EXL3 checkpoint has this library do, as cases that can be timed.

Kinds (each through the public operator of mlxl3_amd):
  linear  Exl3Linear.forward       one projection
  group   Exl3Group.forward        projections of one input (q/k/v)
  mlp     Exl3Mlp.forward          the dense SwiGLU MLP of a decoder layer
  moe     Exl3SwitchGlu.forward    the expert block of a mixture-of-experts layer
  layers  the projections of a stack of decoder layers, one after another

Rows are tokens: 1 in plain decode, 2 to 16 when a batch or a speculative draft is
verified, tens to thousands in prefill.  Weights are random trellis words (every word
is a valid trellis), scales are f16 of +-U(0.5, 1.5) with the output scales carrying
1/sqrt(inputs) as a quantized checkpoint's do, activations N(0, 1) with 1 % of the
channels 20 times larger, routes the top k of softmax(N(0, 1)).
"""

from __future__ import annotations

import math

import torch

import mlxl3_amd

_DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # the key or value projection of one decoded token: the smallest call there is
        dict(name="kv_m1", kind="linear", rows=1, inp=4096, out=1024, k=4, cb=0, dtype="f16", bias=False),
        # an MLP projection of one decoded token
        dict(name="up_m1", kind="linear", rows=1, inp=4096, out=14336, k=4, cb=0, dtype="f16", bias=False),
        # the vocabulary head of one decoded token, at the higher width heads are stored with
        dict(name="head_m1", kind="linear", rows=1, inp=4096, out=151936, k=6, cb=0, dtype="f16", bias=False),
        # q, k and v of a short speculative draft
        dict(name="qkv_m4", kind="group", rows=4, inp=5120, outs="5120,1024,1024", k=3, cb=1, dtype="f16"),
        # the MLP of a wider layer when eight drafted tokens are verified
        dict(name="mlp_m8", kind="mlp", rows=8, inp=5120, hidden=27648, k=2, cb=1),
        # four layers of one decoded token: every projection of them in order
        dict(name="layers_m1", kind="layers", rows=1, layers=4, inp=4096, kv=1024, hidden=14336, k=4, cb=0),
        # a short prompt (or the ragged end of a long one), bfloat16 with a bias
        dict(name="down_m47", kind="linear", rows=47, inp=14336, out=4096, k=5, cb=2, dtype="bf16", bias=True),
        # a prefill chunk through one projection
        dict(name="up_m512", kind="linear", rows=512, inp=4096, out=14336, k=4, cb=0, dtype="f16", bias=False),
        # a long prefill chunk through the MLP
        dict(name="mlp_m2048", kind="mlp", rows=2048, inp=4096, hidden=14336, k=4, cb=0),
        # the experts of one decoded token, of a batch of short chunks, of a long prompt
        dict(name="moe_m1", kind="moe", rows=1, inp=2048, hidden=768, experts=128, top=8, k=3, cb=0,
             dtype="f16", scores="f16", act="silu"),
        dict(name="moe_m256", kind="moe", rows=256, inp=2048, hidden=768, experts=128, top=8, k=3, cb=0,
             dtype="f16", scores="f16", act="silu"),
        dict(name="moe_m2000", kind="moe", rows=2000, inp=2048, hidden=768, experts=128, top=8, k=3, cb=0,
             dtype="f16", scores="f16", act="silu"),
    ]


# ---------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------
_MAX_FLOPS = 7.0e11  # below the largest listed case
_MAX_MOE_FLOPS = 1.5e11  # grouped rows run at a lower rate
_WIDTHS = [(4096, 14336), (14336, 4096), (4096, 4096), (4096, 1024), (5120, 27648), (27648, 5120),
           (5120, 5120), (5120, 1024), (2048, 1536)]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(rng, most):
    """Row counts over the whole range; odd ones as likely as round ones."""
    return max(1, min(_log_int(rng, 1, 4096), int(most)))


def _width(rng, lo, hi):
    return 128 * _log_int(rng, lo // 128, hi // 128)


def _bits(rng):
    return rng.choice([2, 3, 3, 4, 4, 4, 5, 6, 8])


def draw(rng):
    kind = rng.choice(["linear", "linear", "group", "mlp", "moe", "moe", "layers"])
    k, cb = _bits(rng), rng.choice([0, 0, 1, 2])
    if kind == "linear":
        inp, out = rng.choice(_WIDTHS) if rng.random() < 0.5 else (_width(rng, 1024, 28672), _width(rng, 512, 28672))
        rows = _rows(rng, _MAX_FLOPS / (2.0 * inp * out))
        return dict(kind=kind, rows=rows, inp=inp, out=out, k=k, cb=cb,
                    dtype=rng.choice(["f16", "f16", "bf16", "f32"]), bias=rng.random() < 0.25)
    if kind == "group":
        inp, kv = rng.choice([2048, 4096, 5120, _width(rng, 1024, 8192)]), rng.choice([512, 1024, 2048])
        out = rng.choice([inp, _width(rng, 1024, 8192)])
        rows = _rows(rng, _MAX_FLOPS / (2.0 * inp * (out + 2 * kv)))
        return dict(kind=kind, rows=rows, inp=inp, outs="%d,%d,%d" % (out, kv, kv), k=k, cb=cb,
                    dtype=rng.choice(["f16", "f16", "bf16"]))
    if kind == "mlp":
        inp, hidden = rng.choice([(4096, 14336), (5120, 27648), (_width(rng, 1024, 6144), _width(rng, 2048, 20480))])
        return dict(kind=kind, rows=_rows(rng, _MAX_FLOPS / (6.0 * inp * hidden)), inp=inp, hidden=hidden, k=k, cb=cb)
    if kind == "moe":
        inp, hidden = rng.choice([(2048, 768), (2048, 1024), (_width(rng, 1024, 4096), _width(rng, 512, 2048))])
        experts, top = rng.choice([(128, 8), (64, 6), (32, 4), (8, 2)])
        return dict(kind=kind, rows=_rows(rng, _MAX_MOE_FLOPS / (6.0 * inp * hidden * top)), inp=inp, hidden=hidden,
                    experts=experts, top=top, k=k, cb=cb, dtype=rng.choice(["f16", "f16", "bf16"]),
                    scores=rng.choice(["f16", "f16", "f32"]), act=rng.choice(["silu", "silu", "silu", "gelu"]))
    layers, inp, hidden = rng.choice([(4, 4096, 14336), (3, 2048, 6144), (2, 5120, 27648)])
    return dict(kind=kind, rows=_log_int(rng, 1, 32), layers=layers, inp=inp, kv=1024, hidden=hidden, k=k, cb=cb)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _trellis(g, rows, cols, k):
    return torch.randint(-32768, 32768, (rows // 16, cols // 16, 16 * k), dtype=torch.int16, device="cuda", generator=g)


def _scales(g, *shape, gain=1.0):
    u = torch.rand(*shape, device="cuda", generator=g)
    s = torch.rand(*shape, device="cuda", generator=g) < 0.5
    return (torch.where(s, u + 0.5, -0.5 - u) * gain).to(torch.float16)


def _activations(g, rows, width, dtype, outliers=True):
    x = torch.randn(rows, width, device="cuda", generator=g)
    if outliers:
        at = torch.randperm(width, device="cuda", generator=g)[: round(width * 0.01)]
        x[:, at] *= 20.0
    return x.to(_DTYPES[dtype])


def _weights(g, inp, out, k, bias=False, gain=1.0):
    """Trellis, input scales, output scales and bias of one projection."""
    t = _trellis(g, inp, out, k)
    return t, _scales(g, inp), _scales(g, out, gain=gain / math.sqrt(inp)), _scales(g, out) if bias else None


def _inputs(case, seed):
    """Plain tensors of the case: what exact() reads and prepare() hands to the library."""
    g, k, kind = _generator(seed), case["k"], case["kind"]
    if kind == "linear":
        return _weights(g, case["inp"], case["out"], k, case["bias"]), _activations(g, case["rows"], case["inp"], case["dtype"])
    if kind == "group":
        parts = [_weights(g, case["inp"], int(o), k) for o in case["outs"].split(",")]
        return parts, _activations(g, case["rows"], case["inp"], case["dtype"])
    if kind == "mlp":
        i, h = case["inp"], case["hidden"]
        parts = [_weights(g, i, h, k), _weights(g, i, h, k), _weights(g, h, i, k)]
        return parts, _activations(g, case["rows"], i, "f16", outliers=False)
    if kind == "layers":
        i, h, kv = case["inp"], case["hidden"], case["kv"]
        stack = []
        for _ in range(case["layers"]):  # q, k, v, o, gate, up, down; the residual branches end small
            dims = [(i, i, 1.0), (i, kv, 1.0), (i, kv, 1.0), (i, i, 0.1), (i, h, 1.0), (i, h, 1.0), (h, i, 0.1)]
            stack.append([_weights(g, a, b, k, gain=gain) for a, b, gain in dims])
        return stack, _activations(g, case["rows"], i, "f16", outliers=False)
    i, h, e = case["inp"], case["hidden"], case["experts"]
    bank = (_trellis(g, i, 2 * e * h, k), _scales(g, e, 2, i), _scales(g, e, 2, h, gain=1.0 / math.sqrt(i)),
            _trellis(g, h, e * i, k), _scales(g, e, h), _scales(g, e, i, gain=1.0 / math.sqrt(h)))
    x = _activations(g, case["rows"], i, case["dtype"], outliers=False)
    p = torch.softmax(torch.randn(case["rows"], e, device="cuda", generator=g), dim=1)
    top, selected = torch.topk(p, case["top"], dim=1)
    return bank, (x, selected.to(torch.int32), (top / top.sum(1, keepdim=True)).to(_DTYPES[case["scores"]]))


def prepare(case, seed):
    weights, x = _inputs(case, seed)
    k, cb, kind = case["k"], case["cb"], case["kind"]
    lin = lambda w: mlxl3_amd.Exl3Linear(*w, k=k, cb=cb)  # noqa: E731
    if kind == "linear":
        return {"kind": kind, "op": lin(weights), "x": x}
    if kind == "group":
        return {"kind": kind, "op": mlxl3_amd.Exl3Group([lin(w) for w in weights]), "x": x}
    if kind == "mlp":
        return {"kind": kind, "op": mlxl3_amd.Exl3Mlp(*(lin(w) for w in weights)), "x": x}
    if kind == "layers":
        stack = []
        for ws in weights:
            q, kk, v, o, gate, up, down = (lin(w) for w in ws)
            stack.append((mlxl3_amd.Exl3Group([q, kk, v]), o, mlxl3_amd.Exl3Mlp(gate, up, down)))
        return {"kind": kind, "op": stack, "x": x}
    op = mlxl3_amd.Exl3SwitchGlu(*weights, top_k=case["top"], k=k, cb=cb, activation=case["act"])
    return {"kind": kind, "op": op, "x": x}


def run(state):
    kind, op, x = state["kind"], state["op"], state["x"]
    if kind == "moe":
        return op.forward(*x)
    if kind != "layers":
        return op.forward(x)
    # the projections of each layer with the residual sums between them; q stands for the
    # attention's output, which is no work of this library
    out = []
    for qkv, o, mlp in op:
        q, k, v = qkv.forward(x)
        x = x + o.forward(q)
        x = x + mlp.forward(x)
        out += [k, v]
    return [x] + out


def work(case):
    k, kind, rows = case["k"], case["kind"], case["rows"]
    size = {"f16": 2, "bf16": 2, "f32": 4}

    def one(inp, out, n_in=2, n_out=2, bias=False):
        return (inp * out * k / 8 + rows * (inp * n_in + out * n_out) + 2 * inp + 2 * out + (2 * out if bias else 0),
                2.0 * rows * inp * out)

    if kind == "linear":
        n = size[case["dtype"]]
        parts = [one(case["inp"], case["out"], n, 4 if case["bias"] and case["dtype"] == "bf16" else n, case["bias"])]
    elif kind == "group":
        outs = [int(o) for o in case["outs"].split(",")]
        parts = [one(case["inp"], o, 2 if i == 0 else 0) for i, o in enumerate(outs)]  # x is read once
    elif kind == "mlp":  # the hidden activations need not leave the chip
        i, h = case["inp"], case["hidden"]
        parts = [one(i, h, 2, 0), one(i, h, 0, 0), one(h, i, 0, 2)]
    elif kind == "layers":
        i, h, kv, n = case["inp"], case["hidden"], case["kv"], case["layers"]
        layer = [one(i, i, 0, 0), one(i, kv, 0, 2), one(i, kv, 0, 2), one(i, i, 0, 0), one(i, h, 0, 0), one(i, h, 0, 0),
                 one(h, i, 0, 0)]
        parts = layer * n + [(4.0 * rows * i, 0.0)]
    else:
        i, h, e, top = case["inp"], case["hidden"], case["experts"], case["top"]
        # experts that some token is routed to, were every expert as likely
        used = e * (1.0 - (1.0 - top / e) ** rows)
        weights = used * (3 * i * h * k / 8 + 2 * (3 * i + 3 * h))
        n_y = 2 if case["scores"] == "f16" else 4
        io = rows * (i * (2 + n_y) + top * (4 + size[case["scores"]]))
        parts = [(weights + io, 6.0 * rows * top * i * h)]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    """About four times the distance of the path from exact() (its f16 roundings at the
    glue's points; other summation orders move it by less)."""
    rel = {"linear": 2.5e-3, "group": 2.5e-3, "mlp": 5e-3, "moe": 4e-3, "layers": 4e-3}[case["kind"]]
    if case.get("dtype") == "bf16" and case["kind"] in ("linear", "group"):
        rel = 6.5e-3  # the result passes through bfloat16
    return {"rel": rel}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _codewords(cb):
    """The 65536 weights of a codebook, each rounded to f16 once as the format defines them."""
    s = torch.arange(65536, dtype=torch.int64, device="cuda")
    if cb == 2:
        y = (s * 0x83DCD12D) & 0xFFFFFFFF
        n = 0x6400 + (y & 255) + ((y >> 8) & 255) + ((y >> 16) & 255) + (y >> 24)
        half = lambda bits: torch.tensor([bits], dtype=torch.int32, device="cuda").to(torch.uint16).view(torch.float16).double()  # noqa: E731
        h = n.to(torch.int32).to(torch.int16).view(torch.float16).double()
        return (h * half(0x1EEE) + half(0xC931)).half().double()
    y = s * 0xCBAC1FED if cb == 1 else s * 89226354 + 64248484
    y = (y & 0x8FFF8FFF) ^ 0x3B603B60
    half = lambda v: torch.where(v >= 32768, v - 65536, v).to(torch.int16).view(torch.float16).double()  # noqa: E731
    return (half(y & 0xFFFF) + half((y >> 16) & 0xFFFF)).half().double()


def _decode(trellis, k, cb, c0=0, c1=None):
    """[inputs, outputs] weights of tile columns c0..c1 in float64."""
    trellis = trellis[:, c0:c1]
    tr, tc, _ = trellis.shape
    dev = trellis.device
    table = _codewords(cb)
    t = torch.arange(256, device=dev)
    start = ((t + 1) * k - 16) % (256 * k)
    a, off = start >> 5, start & 31
    b = (a + 1) % (8 * k)
    # weight t of a tile: lane t / 32, local state t % 32 = 8p + 4c + 2h + r -> row 8h + 2p + r, column lane + 8c
    j, s = t >> 5, t & 31
    row = 8 * ((s >> 1) & 1) + 2 * (s >> 3) + (s & 1)
    col = j + 8 * ((s >> 2) & 1)
    out = torch.empty(tr * 16, tc * 16, dtype=torch.float64, device=dev)
    place = torch.empty(256, dtype=torch.int64, device=dev)
    place[row * 16 + col] = t
    step = max(1, (1 << 16) // tc)
    for r0 in range(0, tr, step):
        w = trellis[r0:r0 + step].to(torch.int64) & 0xFFFF
        w = w[..., 0::2] | (w[..., 1::2] << 16)
        states = (((w[..., a] << 32) | w[..., b]) >> (48 - off)) & 0xFFFF
        n = w.shape[0]
        tile = table[states][..., place].view(n, tc, 16, 16)
        out[r0 * 16:(r0 + n) * 16] = tile.permute(0, 2, 1, 3).reshape(n * 16, tc * 16)
    return out


def _hadamard(x):
    h = torch.ones(1, 1, dtype=torch.float64, device=x.device)
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x.reshape(-1, 128) @ (h / math.sqrt(128.0))).reshape(x.shape)


def _linear64(w, x, k, cb):
    trellis, suh, svh, bias = w
    xh = _hadamard(x.double() * suh.double())
    step = 4096
    y = torch.cat([xh @ _decode(trellis, k, cb, c, c + step) for c in range(0, trellis.shape[1], step)], 1)
    y = _hadamard(y) * svh.double()
    return y if bias is None else y + bias.double()


def _mlp64(ws, x, k, cb):
    g, u = _linear64(ws[0], x, k, cb), _linear64(ws[1], x, k, cb)
    return _linear64(ws[2], torch.nn.functional.silu(g) * u, k, cb)


def exact(case, seed):
    weights, x = _inputs(case, seed)
    k, cb, kind = case["k"], case["cb"], case["kind"]
    if kind == "linear":
        return _linear64(weights, x, k, cb)
    if kind == "group":
        return [_linear64(w, x, k, cb) for w in weights]
    if kind == "mlp":
        return _mlp64(weights, x, k, cb)
    if kind == "layers":
        out, x = [], x.double()
        for ws in weights:
            out += [_linear64(ws[1], x, k, cb), _linear64(ws[2], x, k, cb)]
            x = x + _linear64(ws[3], _linear64(ws[0], x, k, cb), k, cb)
            x = x + _mlp64(ws[4:], x, k, cb)
        return [x] + out
    gu, gu_suh, gu_svh, down, down_suh, down_svh = weights
    x, selected, scores = x
    i, h, e, top = case["inp"], case["hidden"], case["experts"], case["top"]
    y = torch.zeros(case["rows"], i, dtype=torch.float64, device=x.device)
    for n in range(e):
        token, slot = torch.nonzero(selected == n, as_tuple=True)
        if not token.numel():
            continue
        xe = x[token].half()  # the operator reads its input as f16
        g, u = (_linear64((gu[:, c * h // 16:(c + 1) * h // 16], gu_suh[n, p], gu_svh[n, p], None), xe, k, cb)
                for p, c in ((0, n), (1, e + n)))
        a = (torch.nn.functional.gelu(g, approximate="tanh") if case["act"] == "gelu" else torch.nn.functional.silu(g)) * u
        d = _linear64((down[:, n * i // 16:(n + 1) * i // 16], down_suh[n], down_svh[n], None), a, k, cb)
        y.index_add_(0, token, d * scores[token, slot].double()[:, None])
    return y
