"""Performance cases of the quantized-matmul library.

A case is what a program that runs (or fine-tunes) a model on MLX-packed
weights has this library do in one go:

  step      the quantized linear layers of `layers` transformer blocks over
            `tokens` rows (q, k, v, o, gate, up, down), preceded by the
            embedding lookup and followed by the vocabulary projection where
            `vocab` is set: one row is a decode step, a few rows a batched
            decode or a short prompt, many rows a prefill;
  experts   one routed-expert block: router top-k and sort, the gate, up and
            down projections of the chosen experts, the weighted combine;
  backward  the gradient of a block's linear layers with respect to their
            inputs (dX = dY . W, the transpose=false form), as adapter
            training through frozen quantized weights runs it.

`graph` cases replay a captured graph, as decode loops do; the others encode
every op on each pass.  Attention, norms and activation functions belong to
the program, so every projection has an input of its own here.

Weights: uniform packed values, scales U(0.002, 0.02), biases
-2^(bits-1) * scale + N(0, 1e-3); activations N(0, 1); router logits N(0, 1).
"""
import math

import torch

from cider_press_amd.kernels import Device, KernelLibrary
from cider_press_amd.kernels import embed as kembed
from cider_press_amd.kernels import gather as kgather
from cider_press_amd.kernels import moe as kmoe
from cider_press_amd.kernels import qmm as kqmm
from cider_press_amd.kernels import qmv as kqmv

TORCH_T = {"bf16": torch.bfloat16, "f16": torch.float16}


# --------------------------------------------------------------------------
# Cases
# --------------------------------------------------------------------------

def _step(name, tokens, layers, hidden, kv, inter, vocab=0, bits=4, gs=64, dtype="bf16", graph=False):
    return {"name": name, "kind": "step", "tokens": tokens, "layers": layers, "hidden": hidden, "kv": kv,
            "inter": inter, "vocab": vocab, "bits": bits, "gs": gs, "dtype": dtype, "graph": graph}


def _experts(name, tokens, experts, top_k, hidden, width, bits=4, gs=64, dtype="bf16", graph=False):
    return {"name": name, "kind": "experts", "tokens": tokens, "experts": experts, "top_k": top_k, "hidden": hidden,
            "width": width, "bits": bits, "gs": gs, "dtype": dtype, "graph": graph}


def _backward(name, tokens, hidden, kv, inter, bits=4, gs=64, dtype="bf16"):
    return {"name": name, "kind": "backward", "tokens": tokens, "hidden": hidden, "kv": kv, "inter": inter,
            "bits": bits, "gs": gs, "dtype": dtype}


def listed():
    return [
        # One decode token of a small model (Qwen2.5-0.5B shapes): four of its
        # blocks, the embedding row and the vocabulary projection, replayed as
        # a graph.  Launch and latency bound.
        _step("decode_small", 1, 4, 896, 128, 4864, vocab=151936, graph=True),
        # The same blocks called op by op, as a program without a graph does.
        _step("decode_small_eager", 1, 1, 896, 128, 4864, dtype="f16"),
        # One decode token of a mid-size model: the weight stream.
        _step("decode_large", 1, 3, 4096, 1024, 12288, graph=True),
        # One decode token at a width that does not divide a word.
        _step("decode_sixbit", 1, 6, 2048, 512, 6144, bits=6, graph=True),
        # Eight sequences decoded together, 8-bit weights.
        _step("batch_eightbit", 8, 2, 4096, 1024, 12288, bits=8, graph=True),
        # A short prompt of a small model (39 tokens, the reference's own
        # benchmark length), with its vocabulary projection.
        _step("prompt_39", 39, 2, 896, 128, 4864, vocab=151936),
        # A prefill chunk.
        _step("prefill_512", 512, 1, 4096, 1024, 12288),
        # A long prefill, for sustained matrix-core throughput.
        _step("prefill_2048", 2048, 1, 4096, 1024, 12288),
        # A prompt of odd length with 8-bit weights in small groups, fp16.
        _step("prefill_eightbit", 777, 1, 4096, 1024, 12288, bits=8, gs=32, dtype="f16"),
        # Routed experts: four tokens decoded together.
        _experts("experts_decode", 4, 128, 8, 2048, 768, graph=True),
        # Routed experts: a 256-token prefill.
        _experts("experts_prefill", 256, 128, 8, 2048, 768),
        # Adapter training through one frozen block.
        _backward("backward_512", 512, 4096, 1024, 12288),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _multiple(v, of, lo):
    return max(lo, int(v) // of * of)


def draw(rng):
    """A case of the same ranges: decode, batched decode, prefill, routed
    experts, backward; model widths over the range small to large, multiples
    of the group size only (so odd multiples are frequent)."""
    what = rng.choices(["decode", "batch", "prefill", "experts", "backward"], weights=[6, 5, 5, 4, 3])[0]
    gs = rng.choice([32, 64, 64, 64, 128])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    if what == "experts":
        unit = max(gs, 32)
        tokens = int(_log_uniform(rng, 1, 513))
        experts = rng.choice([8, 16, 32, 64, 96, 128])
        hidden = _multiple(_log_uniform(rng, 512, 4096), 128, 512)
        width = _multiple(_log_uniform(rng, 384, 2048), 128, 384)
        return {k: v for k, v in _experts("", tokens, experts, rng.choice([2, 4, 6, 8]), hidden, width,
                                          bits=rng.choice([4, 4, 8]), gs=unit, dtype=dtype,
                                          graph=tokens <= 8).items() if k != "name"}
    bits = rng.choice([4, 4, 4, 4, 8, 8, 6, 3])
    unit = max(gs, 64)
    hidden = _multiple(_log_uniform(rng, 512, 5200), unit, 512)
    kv = _multiple(hidden / rng.choice([1, 4, 7, 8]), unit, unit)
    inter = _multiple(hidden * rng.uniform(2.0, 4.0), unit, 1024)
    if what == "backward":
        tokens = int(_log_uniform(rng, 16, 1024))
        c = _backward("", tokens, hidden, kv, inter, bits=bits, gs=gs, dtype=dtype)
    else:
        lo, hi = {"decode": (1, 2), "batch": (2, 65), "prefill": (65, 2049)}[what]
        tokens = 1 if what == "decode" else int(_log_uniform(rng, lo, hi))
        layers = rng.randint(1, 4) if tokens <= 64 else 1
        vocab = rng.choice([0, 0, 32000]) if tokens <= 64 else 0
        if bits in (3, 6):  # widths that straddle words: the prefill range that costs no more than the largest case
            tokens = min(tokens, 512)
        c = _step("", tokens, layers, hidden, kv, inter, vocab=vocab, bits=bits, gs=gs, dtype=dtype,
                  graph=tokens <= 16 and rng.random() < 0.8)
    del c["name"]
    # No drawn case costs more than the largest listed one.
    limit = 2.0 * 2048 * (2 * 4096 * 4096 + 2 * 1024 * 4096 + 3 * 4096 * 12288)
    limit *= {4: 0.8, 8: 0.4}.get(bits, 0.15) if what != "backward" else 0.15
    flops = work(c)["flops"]
    if flops > limit:
        c["tokens"] = max(1, int(c["tokens"] * limit / flops))
    return c


# --------------------------------------------------------------------------
# Shapes of a case
# --------------------------------------------------------------------------

def _projections(c):
    """(label, rows in N, columns in K, input label) of one block."""
    h, kv, i = c["hidden"], c["kv"], c["inter"]
    return [("q", h, h, "attn_in"), ("k", kv, h, "attn_in"), ("v", kv, h, "attn_in"), ("o", h, h, "attn_out"),
            ("gate", i, h, "mlp_in"), ("up", i, h, "mlp_in"), ("down", h, i, "mlp_act")]


def _weight_bytes(c, n, k):
    return n * k * c["bits"] // 8 + 2 * n * (k // c["gs"]) * 2


def work(case):
    """Bytes and operations a pass cannot do without."""
    c, m = case, case["tokens"]
    if c["kind"] == "experts":
        rows = m * c["top_k"]
        touched = c["experts"] * (1.0 - (1.0 - c["top_k"] / c["experts"]) ** m)
        per = 2 * _weight_bytes(c, c["width"], c["hidden"]) + _weight_bytes(c, c["hidden"], c["width"])
        io = 2 * (m * c["hidden"] + 2 * rows * c["width"] + rows * c["width"] + 2 * rows * c["hidden"] +
                  m * c["hidden"] + m * c["experts"]) + 6 * rows * 4
        return {"bytes": touched * per + io, "flops": 2.0 * rows * 3 * c["width"] * c["hidden"]}
    proj = _projections(c)
    if c["kind"] == "backward":
        return {"bytes": sum(_weight_bytes(c, n, k) + 2 * m * (n + k) for _, n, k, _ in proj),
                "flops": sum(2.0 * m * n * k for _, n, k, _ in proj)}
    inputs = 2 * m * (3 * c["hidden"] + c["inter"])
    nbytes = c["layers"] * (sum(_weight_bytes(c, n, k) + 2 * m * n for _, n, k, _ in proj) + inputs)
    flops = c["layers"] * sum(2.0 * m * n * k for _, n, k, _ in proj)
    if c["vocab"]:
        nbytes += _weight_bytes(c, c["vocab"], c["hidden"]) + 2 * m * (c["vocab"] + c["hidden"])
        nbytes += m * (4 + _weight_bytes(c, 1, c["hidden"]) + 2 * c["hidden"])
        flops += 2.0 * m * c["vocab"] * c["hidden"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the error of one correctly rounded 16-bit output
    against 64 bits (1.7e-3 in bf16, 2.1e-4 in f16, measured); the largest
    single difference is a few roundings at the largest outputs."""
    return {"rel": 7e-3, "max": 6e-2} if case["dtype"] == "bf16" else {"rel": 9e-4, "max": 8e-3}


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------

_PROGRAM = {}  # the device, kernel library and command session of this program


def _program():
    if not _PROGRAM:
        dev = Device.system_default()
        _PROGRAM.update(dev=dev, lib=KernelLibrary.quantized(dev), cmds=dev.commands())
    return _PROGRAM["dev"], _PROGRAM["lib"], _PROGRAM["cmds"]


class _Memory:
    """A library buffer as torch sees it."""

    TYPES = {"bf16": "<u2", "f16": "<u2", "u32": "<i4", "f32": "<f4"}

    def __init__(self, buf):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": (len(buf),), "typestr": self.TYPES[buf.dtype],
                                         "data": (buf.ptr, False), "strides": None, "version": 2}


def _view(buf, *shape):
    t = torch.as_tensor(_Memory(buf), device="cuda")
    if buf.dtype in TORCH_T:
        t = t.view(TORCH_T[buf.dtype])
    return t.reshape(shape) if shape else t


class _Values:
    """The case's input values as torch tensors, a function of the seed alone."""

    def __init__(self, case, seed):
        self.c = case
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def weight(self, n, k):
        c, t = self.c, TORCH_T[self.c["dtype"]]
        words = torch.randint(-2**31, 2**31, (n, k * c["bits"] // 32), dtype=torch.int32, device="cuda",
                              generator=self.g)
        s = torch.empty(n, k // c["gs"], device="cuda").uniform_(0.002, 0.02, generator=self.g).to(t)
        noise = torch.empty_like(s, dtype=torch.float32).normal_(0.0, 1e-3, generator=self.g)
        b = (-float(1 << (c["bits"] - 1)) * s.float() + noise).to(t)
        return words, s, b

    def x(self, m, k):
        return torch.empty(m, k, device="cuda").normal_(0.0, 1.0, generator=self.g).to(TORCH_T[self.c["dtype"]])

    def ids(self, n, below):
        return torch.randint(0, below, (n,), dtype=torch.int32, device="cuda", generator=self.g)


def _values(case, seed):
    """{label: tensor or (words, scales, biases)}, in one fixed order."""
    c, m, v, out = case, case["tokens"], _Values(case, seed), {}
    if c["kind"] == "experts":
        e, h, w = c["experts"], c["hidden"], c["width"]
        out["logits"], out["x"] = v.x(m, e), v.x(m, h)
        out["act"] = v.x(m * c["top_k"], w)
        out["gate"], out["up"], out["down"] = v.weight(e * w, h), v.weight(e * w, h), v.weight(e * h, w)
        return out
    if c["kind"] == "backward":
        for label, n, k, _ in _projections(c):
            out[label], out["d" + label] = v.weight(n, k), v.x(m, n)
        return out
    if c["vocab"]:
        out["ids"], out["table"] = v.ids(m, c["vocab"]), v.weight(c["vocab"], c["hidden"])
        out["head_in"] = v.x(m, c["hidden"])
    for layer in range(c["layers"]):
        for label, width in (("attn_in", "hidden"), ("attn_out", "hidden"), ("mlp_in", "hidden"),
                             ("mlp_act", "inter")):
            out["%d.%s" % (layer, label)] = v.x(m, c[width])
        for label, n, k, _ in _projections(c):
            out["%d.%s" % (layer, label)] = v.weight(n, k)
    return out


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------

def prepare(case, seed):
    dev, _, cmds = _program()
    c, m = case, case["tokens"]
    buf, out = {}, {}

    def load(t, dtype):
        b = dev.alloc_buffer(t.numel(), dtype)
        _view(b).copy_(t.reshape(-1))
        return b

    for label, v in _values(case, seed).items():
        if isinstance(v, tuple):
            buf[label] = (load(v[0], "u32"), load(v[1], c["dtype"]), load(v[2], c["dtype"]))
        else:
            buf[label] = load(v, "u32" if v.dtype == torch.int32 else c["dtype"])
        del v

    def output(label, dtype, *shape):
        buf["out." + label] = dev.alloc_buffer(math.prod(shape), dtype)
        out[label] = _view(buf["out." + label], *shape).zero_()

    if c["kind"] == "experts":
        rows = m * c["top_k"]
        for label in ("experts", "lhs", "rhs", "inv"):
            output(label, "u32", rows)
        output("offsets", "u32", c["experts"] + 1)
        output("scores", "f32", m, c["top_k"])
        output("gate", c["dtype"], rows, c["width"])
        output("up", c["dtype"], rows, c["width"])
        output("down", c["dtype"], rows, c["hidden"])
        output("y", c["dtype"], m, c["hidden"])
    elif c["kind"] == "backward":
        for label, n, k, _ in _projections(c):
            output(label, c["dtype"], m, k)
    else:
        if c["vocab"]:
            output("embedded", c["dtype"], m, c["hidden"])
        for layer in range(c["layers"]):
            for label, n, k, _ in _projections(c):
                output("%d.%s" % (layer, label), c["dtype"], m, n)
        if c["vocab"]:
            output("logits", c["dtype"], m, c["vocab"])
    state = {"case": c, "buf": buf, "out": out, "graph": None}
    if c.get("graph"):
        torch.cuda.synchronize()
        _encode(state)  # warm up, then record
        cmds.commit_and_wait()
        cmds.begin_capture()
        _encode(state)
        state["graph"] = cmds.end_capture()
        for t in out.values():
            t.zero_()
    return state


def _encode(state):
    _, lib, cmds = _program()
    c, buf = state["case"], state["buf"]
    m, gs, bits = c["tokens"], c["gs"], c["bits"]

    if c["kind"] == "experts":
        e, h, w, rows = c["experts"], c["hidden"], c["width"], c["tokens"] * c["top_k"]
        kmoe.moe_route(cmds, buf["logits"], m, e, c["top_k"], True, buf["out.experts"], buf["out.scores"],
                       buf["out.lhs"], buf["out.rhs"], buf["out.inv"], buf["out.offsets"])
        for label in ("gate", "up"):
            kgather.affine_gather_qmm(cmds, lib, buf["x"], *buf[label], buf["out.lhs"], buf["out.rhs"],
                                      buf["out." + label], rows, w, h, e, gs, bits, sorted_indices=True)
        kgather.affine_gather_qmm(cmds, lib, buf["act"], *buf["down"], None, buf["out.rhs"], buf["out.down"], rows,
                                  h, w, e, gs, bits, sorted_indices=True)
        kmoe.moe_combine(cmds, buf["out.down"], buf["out.scores"], buf["out.inv"], m, c["top_k"], h, buf["out.y"])
        return

    if c["kind"] == "backward":
        for label, n, k, _ in _projections(c):
            kqmm.affine_qmm_n(cmds, lib, *buf[label], buf["d" + label], buf["out." + label], m, k, n, gs, bits)
        return

    def linear(weight, x, y, n, k):
        if m == 1:
            kqmv.affine_qmv(cmds, lib, *weight, x, y, k, gs, bits)
        else:
            kqmm.affine_qmm_t(cmds, lib, *weight, x, y, m, n, k, gs, bits)

    if c["vocab"]:
        kembed.embed_tokens(cmds, lib, *buf["table"], buf["ids"], buf["out.embedded"], c["vocab"], c["hidden"], gs,
                            bits)
    for layer in range(c["layers"]):
        for label, n, k, source in _projections(c):
            linear(buf["%d.%s" % (layer, label)], buf["%d.%s" % (layer, source)], buf["out.%d.%s" % (layer, label)],
                   n, k)
    if c["vocab"]:
        linear(buf["table"], buf["head_in"], buf["out.logits"], c["vocab"], c["hidden"])


def run(state):
    if state["graph"] is not None:
        state["graph"].launch(_program()[2])
    else:
        _encode(state)
    return state["out"]


# --------------------------------------------------------------------------
# The same values in 64 bits
# --------------------------------------------------------------------------

def _dequantized(c, weight):
    """The weight as the format defines it: fmaf(scale, q, bias) rounded to T."""
    words, s, b = weight
    bits, gs, t = c["bits"], c["gs"], TORCH_T[c["dtype"]]
    n, k = words.shape[0], words.shape[1] * 32 // bits
    u = (words.to(torch.int64) & 0xFFFFFFFF).reshape(n, k // 32, bits)
    q = torch.empty(n, k // 32, 32, dtype=torch.float64, device=words.device)
    for i in range(32):
        at, off = i * bits // 32, i * bits % 32
        v = u[:, :, at] >> off
        if off + bits > 32:
            v = v | (u[:, :, at + 1] << (32 - off))
        q[:, :, i] = (v & ((1 << bits) - 1)).to(torch.float64)
    q = q.reshape(n, k // gs, gs)
    return (q * s.double()[:, :, None] + b.double()[:, :, None]).float().to(t).double().reshape(n, k)


def exact(case, seed):
    c, m, v = case, case["tokens"], _values(case, seed)
    if c["kind"] == "backward":
        return {label: v["d" + label].double() @ _dequantized(c, v[label]) for label, _, _, _ in _projections(c)}
    if c["kind"] == "step":
        out = {}
        for layer in range(c["layers"]):
            for label, n, k, source in _projections(c):
                w = _dequantized(c, v["%d.%s" % (layer, label)])
                out["%d.%s" % (layer, label)] = v["%d.%s" % (layer, source)].double() @ w.t()
        if c["vocab"]:
            w = _dequantized(c, v["table"])
            out["embedded"] = w[v["ids"].long()]
            out["logits"] = v["head_in"].double() @ w.t()
        return out
    e, top, h, w = c["experts"], c["top_k"], c["hidden"], c["width"]
    # Largest probability first, the lower expert among equals.
    p = torch.softmax(v["logits"].double(), dim=1)
    chosen = torch.sort(v["logits"].double(), dim=1, descending=True, stable=True).indices[:, :top]
    scores = torch.gather(p, 1, chosen)
    scores = scores / scores.sum(dim=1, keepdim=True)
    flat = chosen.reshape(-1)
    order = torch.sort(flat, stable=True).indices  # rows by expert
    inv = torch.empty_like(order)
    inv[order] = torch.arange(order.numel(), device=order.device)
    token, expert = order // top, flat[order]
    out = {"scores": scores, "experts": None, "lhs": None, "rhs": None, "inv": None, "offsets": None}
    xs = {"gate": v["x"].double()[token], "up": v["x"].double()[token], "down": v["act"].double()}
    for label, n in (("gate", w), ("up", w), ("down", h)):
        k = xs[label].shape[1]
        words, s, b = (t.reshape(e, n, -1) for t in v[label])
        out[label] = torch.zeros(expert.numel(), n, dtype=torch.float64, device="cuda")
        for i in torch.unique(expert).tolist():
            rows = torch.nonzero(expert == i).reshape(-1)
            out[label][rows] = xs[label][rows] @ _dequantized(c, (words[i], s[i], b[i])).t()
        assert k % c["gs"] == 0
    # The combine rounds sums of the down projection's rounded outputs.
    down = out["down"].float().to(TORCH_T[c["dtype"]]).double()
    out["y"] = (scores[:, :, None] * down[inv].reshape(m, top, h)).sum(dim=1)
    return out
