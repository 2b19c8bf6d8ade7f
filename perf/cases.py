"""Performance cases: what a QLoRA user has this package do, through its public entry points.

Shapes are those of the Qwen2.5 1.5B and 7B projections, the Qwen2.5-1.5B head and
the packed batches that the tests and the benchmark use; T is the number of packed
tokens.  Kinds of case:

  linear     one frozen NF4 Linear4bit: generation (T = 1 ..), prompt and training
             (output and input gradient) up to 16384 tokens
  decode     the frozen NF4 products of one 7B decoder layer for a few tokens, replayed
             from a HIP graph, as a generation loop with static buffers does
  qlora      one NF4 + LoRA projection, forward and backward, with and without the
             LoRA dropout of 0.05
  mlp        the frozen NF4 MLP node, forward and backward
  attention  causal attention over packed rows, forward and backward
  norm       residual add + RMSNorm, forward and backward
  head       fused linear cross-entropy over the whole vocabulary, with a frozen head
             or with the head's gradient
  dequant    decoding one NF4 weight (merging adapters, calls outside the fused path)
  layer      a whole 1.5B decoder layer training step with LoRA on all seven
             projections, replayed from a HIP graph

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a
program has in hand before the call, run() is one pass, work() its floor in bytes and
flops, tolerance() the bound on two correct results and exact() the result in 64 bits.
"""

import math
from types import SimpleNamespace

import torch

from soupsuck_amd.bnb_compat import Params4bit, QuantState, dequantize_4bit
from soupsuck_amd.bnb_compat import nn as bnn
from soupsuck_amd.kernels.add_rmsnorm import add_rms_norm
from soupsuck_amd.kernels.attention import packed_causal_attention, row_offsets
from soupsuck_amd.kernels.cross_entropy import fused_linear_cross_entropy
from soupsuck_amd.kernels.rmsnorm import rms_norm
from soupsuck_amd.kernels.rope import fused_rope
from soupsuck_amd.kernels.swiglu import swiglu
from soupsuck_amd.lora import qlora_projection
from soupsuck_amd.mlp import fused_qwen2_mlp

HIDDEN, INTER, KV, HEADS, KV_HEADS = 1536, 8960, 256, 12, 2      # Qwen2.5-1.5B
HIDDEN7, INTER7, KV7, HEADS7, KV_HEADS7 = 3584, 18944, 512, 28, 4  # Qwen2.5-7B
VOCAB = 151936
HEAD_DIM = 128
EPS = 1e-6
RANK, SCALING = 16, 2.0


# ----------------------------------------------------------------- the cases

def listed():
    return [
        # one token through the widest frozen projection: interactive generation
        {"name": "linear_t1", "kind": "linear", "t": 1, "n": INTER7, "k": HIDDEN7,
         "grad": False},
        # a small batch of sequences generating together, one 7B layer's seven products
        {"name": "decode_t5", "kind": "decode", "t": 5},
        # a short prompt or micro-batch through the down projection, odd T, both directions
        {"name": "linear_t101", "kind": "linear", "t": 101, "n": HIDDEN7, "k": INTER7,
         "grad": True},
        # an ordinary training batch through a square attention projection of the 7B model
        {"name": "linear_t2048", "kind": "linear", "t": 2048, "n": HIDDEN7, "k": HIDDEN7,
         "grad": True},
        # the largest batch through the widest projection
        {"name": "linear_t16384", "kind": "linear", "t": 16384, "n": INTER7, "k": HIDDEN7,
         "grad": True},
        # LoRA on a frozen gate projection with the default adapter dropout
        {"name": "qlora_t826", "kind": "qlora", "t": 826, "n": INTER, "k": HIDDEN,
         "bias": False, "dropout": 0.05},
        # the MLP of a layer whose adapters sit on q and v only
        {"name": "mlp_t990", "kind": "mlp", "t": 990, "hidden": HIDDEN, "inter": INTER},
        # longer documents packed together, 7B heads
        {"name": "attention_t6041", "kind": "attention", "heads": HEADS7,
         "kv_heads": KV_HEADS7, "lengths": "2048,1537,1201,777,350,128"},
        # the norm between attention and MLP with a trained weight, a large batch
        {"name": "norm_t16384", "kind": "norm", "t": 16384, "h": HIDDEN, "train_weight": True},
        # loss and gradients of the tied head, the batch of a real step
        {"name": "head_t826", "kind": "head", "t": 826, "weight_grad": True},
        # decoding the widest weight
        {"name": "dequant_7b", "kind": "dequant", "n": INTER7, "k": HIDDEN7},
        # one layer of a training step on a packed batch of four rows
        {"name": "layer_t990", "kind": "layer", "lengths": "382,242,208,158"},
    ]


def _spread(rng, low, high):
    """A whole number of [low, high], uniform over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


_SHAPES = ((HIDDEN, HIDDEN), (KV, HIDDEN), (INTER, HIDDEN), (HIDDEN, INTER),
           (HIDDEN7, HIDDEN7), (KV7, HIDDEN7), (INTER7, HIDDEN7), (HIDDEN7, INTER7))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "decode", "qlora", "qlora", "mlp",
                       "attention", "norm", "head", "dequant", "layer", "layer"))
    if kind == "linear":
        n, k = rng.choice(_SHAPES)
        return {"kind": kind, "t": _spread(rng, 1, 16384), "n": n, "k": k,
                "grad": rng.random() < 0.6}
    if kind == "decode":
        return {"kind": kind, "t": _spread(rng, 1, 32)}
    if kind == "qlora":
        n, k = rng.choice(_SHAPES)
        return {"kind": kind, "t": _spread(rng, 64, 4096), "n": n, "k": k,
                "bias": rng.random() < 0.5, "dropout": rng.choice((0.0, 0.05))}
    if kind == "mlp":
        hidden, inter = rng.choice(((HIDDEN, INTER), (HIDDEN, INTER), (HIDDEN7, INTER7)))
        return {"kind": kind, "t": _spread(rng, 64, 4096), "hidden": hidden, "inter": inter}
    if kind == "attention":
        heads, kv = rng.choice(((HEADS, KV_HEADS), (HEADS7, KV_HEADS7)))
        lengths, total = [], _spread(rng, 300, 6000)
        while sum(lengths) < total:
            lengths.append(min(_spread(rng, 17, 2048), total - sum(lengths)))
        return {"kind": kind, "heads": heads, "kv_heads": kv,
                "lengths": ",".join(map(str, lengths))}
    if kind == "norm":
        return {"kind": kind, "t": _spread(rng, 128, 16384), "h": rng.choice((HIDDEN, HIDDEN7)),
                "train_weight": rng.random() < 0.5}
    if kind == "head":
        return {"kind": kind, "t": _spread(rng, 128, 1600), "weight_grad": rng.random() < 0.4}
    if kind == "dequant":
        n, k = rng.choice(_SHAPES)
        return {"kind": kind, "n": n, "k": k}
    lengths = [rng.randint(80, 400) for _ in range(rng.randint(1, 8))]
    return {"kind": kind, "lengths": ",".join(map(str, lengths))}


# ------------------------------------------------------------- what is in hand

_NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
        -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
        0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
        0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _normal(gen, shape, std=1.0, dtype=torch.float16):
    return torch.randn(shape, generator=gen, device=gen.device, dtype=torch.float32) \
        .mul_(std).to(dtype)


def _code2():
    """The 256 signed values of the second-level statistics (8-bit dynamic map), sorted."""
    values = [0.0, 1.0]
    for i in range(7):
        edges = torch.linspace(0.1, 1.0, 2 ** i + 1, dtype=torch.float32)
        mids = (10.0 ** (i - 6)) * ((edges[:-1] + edges[1:]) / 2.0)
        values += mids.tolist() + (-mids).tolist()
    return torch.tensor(sorted(values), dtype=torch.float32)


def _nearest(values, table):
    return torch.bucketize(values, (table[:-1] + table[1:]) / 2.0, out_int32=True)


def _checkpoint(gen, n, k):
    """A frozen weight as a bitsandbytes checkpoint holds it: NF4 codes in blocks of 64 of
    N(0, 0.02) values with double-quantized block scales (plain torch)."""
    dev = gen.device
    blocks = _normal(gen, (n * k // 64, 64), 0.02).float()
    absmax = blocks.abs().amax(1)
    nf4 = torch.tensor(_NF4, device=dev)
    codes = _nearest(blocks.div_(absmax[:, None]), nf4).to(torch.uint8).view(-1, 2)
    packed = ((codes[:, 0] << 4) | codes[:, 1]).view(-1, 1)
    code2 = _code2().to(dev)
    offset = absmax.mean().reshape(1)
    rest = absmax - offset
    padded = torch.nn.functional.pad(rest, (0, -rest.numel() % 256)).view(-1, 256)
    absmax2 = padded.abs().amax(1)
    qabs = _nearest((padded / absmax2[:, None]).view(-1)[:rest.numel()], code2).to(torch.uint8)
    return {"n": n, "k": k, "packed": packed, "absmax": qabs, "absmax2": absmax2,
            "code2": code2, "nf4": nf4, "offset": offset}


def _weight(ck):
    """(packed codes, QuantState) of a checkpoint weight."""
    state2 = QuantState(ck["absmax2"], code=ck["code2"], blocksize=256, dtype=torch.float32)
    state = QuantState(ck["absmax"], shape=(ck["n"], ck["k"]), code=ck["nf4"], blocksize=64,
                       quant_type="nf4", dtype=torch.float16, offset=ck["offset"],
                       state2=state2)
    return ck["packed"], state


def _linear(ck):
    """The frozen Linear4bit module of a checkpoint weight."""
    lin = bnn.Linear4bit(ck["k"], ck["n"], bias=False, compute_dtype=torch.float16,
                         device="meta")
    packed, state = _weight(ck)
    lin.weight = Params4bit(packed, quant_state=state)
    return lin


def _decoded(ck):
    """The weight the format defines, fp16 values, in 64 bits (plain torch)."""
    codes = torch.stack((ck["packed"] >> 4, ck["packed"] & 15), -1).view(-1, 64)
    scale = ck["code2"][ck["absmax"].long()] \
        * ck["absmax2"].repeat_interleave(256)[:ck["absmax"].numel()] + ck["offset"]
    w = ck["nf4"][codes.int()] * scale[:, None]
    return w.to(torch.float16).view(ck["n"], ck["k"])


_PROJECTIONS = (("q", HIDDEN, HIDDEN, True), ("k", KV, HIDDEN, True), ("v", KV, HIDDEN, True),
                ("o", HIDDEN, HIDDEN, False), ("gate", INTER, HIDDEN, False),
                ("up", INTER, HIDDEN, False), ("down", HIDDEN, INTER, False))
_DECODE = (("q", HIDDEN7, HIDDEN7), ("k", KV7, HIDDEN7), ("v", KV7, HIDDEN7),
           ("o", HIDDEN7, HIDDEN7), ("gate", INTER7, HIDDEN7), ("up", INTER7, HIDDEN7),
           ("down", HIDDEN7, INTER7))


def _adapter(gen, n, k, bias):
    """LoRA A (Kaiming-uniform), B ~ N(0, 0.01) and the projection's bias."""
    a = (torch.rand((RANK, k), generator=gen, device=gen.device) * 2 - 1) / math.sqrt(k)
    return {"a": a.to(torch.float16), "b": _normal(gen, (n, RANK), 0.01),
            "bias": _normal(gen, (n,), 0.02) if bias else None}


def _lengths(case):
    return [int(v) for v in case["lengths"].split(",")]


def _rope_tables(lengths, dev):
    pos = torch.cat([torch.arange(n, dtype=torch.float64) for n in lengths])
    inv = 1.0 / (1_000_000 ** (torch.arange(0, HEAD_DIM, 2, dtype=torch.float64) / HEAD_DIM))
    ang = pos[:, None] * inv[None, :]
    ang = torch.cat([ang, ang], dim=-1)[None]
    return ang.cos().half().to(dev), ang.sin().half().to(dev)


def _inputs(case, seed):
    """The case's tensors, made from the seed alone with plain torch."""
    kind, gen = case["kind"], _generator(seed)
    if kind in ("linear", "qlora"):
        n, k, t = case["n"], case["k"], case["t"]
        d = {"w": _checkpoint(gen, n, k), "x": _normal(gen, (t, k)),
             "g": _normal(gen, (t, n), 0.01)}
        if kind == "qlora":
            d.update(_adapter(gen, n, k, case["bias"]))
            d["mask_seed"] = int(seed) % (1 << 31)
        return d
    if kind == "decode":
        d = {name: _checkpoint(gen, n, k) for name, n, k in _DECODE}
        for name in ("x", "x_o", "x_mlp"):  # inputs of q / k / v, of o and of the MLP
            d[name] = _normal(gen, (case["t"], HIDDEN7))
        return d
    if kind == "mlp":
        h, i, t = case["hidden"], case["inter"], case["t"]
        return {"gate": _checkpoint(gen, i, h), "up": _checkpoint(gen, i, h),
                "down": _checkpoint(gen, h, i), "x": _normal(gen, (t, h)),
                "g": _normal(gen, (t, h), 0.01)}
    if kind == "attention":
        total = sum(_lengths(case))
        d = {name: _normal(gen, (1, total, heads * HEAD_DIM))
             for name, heads in (("q", case["heads"]), ("k", case["kv_heads"]),
                                 ("v", case["kv_heads"]))}
        d["g"] = _normal(gen, (1, total, case["heads"], HEAD_DIM), 0.01)
        return d
    if kind == "norm":
        shape = (case["t"], case["h"])
        return {"r": _normal(gen, shape), "d": _normal(gen, shape),
                "w": (1 + 0.1 * _normal(gen, shape[1:], 1.0, torch.float32)).half(),
                "gs": _normal(gen, shape, 0.01), "gy": _normal(gen, shape, 0.01)}
    if kind == "head":
        t = case["t"]
        targets = torch.randint(0, VOCAB, (t,), generator=gen, device=gen.device)
        ignored = torch.rand(t, generator=gen, device=gen.device) < 0.365
        return {"x": _normal(gen, (t, HIDDEN)), "w": _normal(gen, (VOCAB, HIDDEN), 0.02),
                "targets": torch.where(ignored, -100, targets)}
    if kind == "dequant":
        return {"w": _checkpoint(gen, case["n"], case["k"])}
    total = sum(_lengths(case))
    d = {"h": _normal(gen, (total, HIDDEN)), "g": _normal(gen, (total, HIDDEN), 0.01)}
    for name in ("norm_in", "norm_post"):
        d[name] = (1 + 0.1 * _normal(gen, (HIDDEN,), 1.0, torch.float32)).half()
    for name, n, k, bias in _PROJECTIONS:
        d[name] = {"w": _checkpoint(gen, n, k), **_adapter(gen, n, k, bias)}
    d["cos"], d["sin"] = _rope_tables(_lengths(case), gen.device)
    return d


_CAPTURE_STREAM = []


def _captured(step):
    """(graph, outputs) of step() after two warm-up runs on the capture stream."""
    if not _CAPTURE_STREAM:
        _CAPTURE_STREAM.append(torch.cuda.Stream())
    side = _CAPTURE_STREAM[0]
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        outs = step()
    return graph, outs


def prepare(case, seed):
    kind, d = case["kind"], _inputs(case, seed)
    s = SimpleNamespace(kind=kind, case=case)
    if kind == "linear":
        s.lin, s.x, s.g = _linear(d["w"]), d["x"].requires_grad_(case["grad"]), d["g"]
    elif kind == "decode":
        lin = {name: _linear(d[name]) for name, _, _ in _DECODE}
        mlp = SimpleNamespace(gate_proj=lin["gate"], up_proj=lin["up"], down_proj=lin["down"])

        def decode():
            with torch.no_grad():
                return (lin["q"](d["x"]), lin["k"](d["x"]), lin["v"](d["x"]),
                        lin["o"](d["x_o"]), fused_qwen2_mlp(mlp, d["x_mlp"]))

        s.keep = d
        s.graph, s.outs = _captured(decode)
    elif kind == "qlora":
        s.packed, s.state = _weight(d["w"])
        s.bias, s.x, s.g, s.mask_seed = d["bias"], d["x"], d["g"], d["mask_seed"]
        s.a, s.b = d["a"], d["b"]
        for t in (s.x, s.a, s.b):
            t.requires_grad_()
    elif kind == "mlp":
        s.mlp = SimpleNamespace(**{name + "_proj": _linear(d[name])
                                   for name in ("gate", "up", "down")})
        s.x, s.g = d["x"].requires_grad_(), d["g"]
    elif kind == "attention":
        s.lengths = _lengths(case)
        s.cu = row_offsets(s.lengths, d["q"].device)
        s.qkv = [d[name].requires_grad_() for name in ("q", "k", "v")]
        s.heads, s.g = (case["heads"], case["kv_heads"], case["kv_heads"]), d["g"]
    elif kind == "norm":
        s.r, s.d = d["r"].requires_grad_(), d["d"].requires_grad_()
        s.w, s.gs, s.gy = d["w"].requires_grad_(case["train_weight"]), d["gs"], d["gy"]
    elif kind == "head":
        s.x, s.targets = d["x"].requires_grad_(), d["targets"]
        s.w = d["w"].requires_grad_(case["weight_grad"])
        s.labelled = (s.targets >= 0).sum().float()
    elif kind == "dequant":
        s.packed, s.state = _weight(d["w"])
    else:
        s.keep, s.lengths = d, _lengths(case)
        s.cu = row_offsets(s.lengths, d["h"].device)
        s.weights = {name: _weight(d[name]["w"]) for name, *_ in _PROJECTIONS}
        s.leaves = [d["h"]] + [d[name][m] for name, *_ in _PROJECTIONS for m in ("a", "b")]
        for t in s.leaves:
            t.requires_grad_()
        s.graph, s.outs = _captured(lambda: _layer_step(s))
    return s


# --------------------------------------------------------------------- one pass

def _layer_step(s):
    """One decoder layer, forward and backward: (output, dH, dA and dB of each projection)."""
    d, total = s.keep, sum(s.lengths)

    def project(name, x):
        p = d[name]
        return qlora_projection(x, p["a"], p["b"], *s.weights[name], p["bias"], SCALING)

    def heads_of(x, heads):
        return x.view(1, total, heads, HEAD_DIM).transpose(1, 2)

    x = rms_norm(d["h"], d["norm_in"], EPS)
    q, k, v = (heads_of(project(name, x), heads)
               for name, heads in (("q", HEADS), ("k", KV_HEADS), ("v", KV_HEADS)))
    q, k = fused_rope(q, k, d["cos"], d["sin"])
    attn = packed_causal_attention(q, k, v, s.lengths, HEAD_DIM ** -0.5, cu_seqlens=s.cu)
    o = project("o", attn.view(total, HIDDEN))
    residual, x = add_rms_norm(d["h"], o, d["norm_post"], EPS)
    out = residual + project("down", swiglu(project("gate", x), project("up", x)))
    return (out.detach(), *torch.autograd.grad(out, s.leaves, d["g"]))


def run(s):
    kind = s.kind
    if kind == "linear":
        if not s.case["grad"]:
            with torch.no_grad():
                return s.lin(s.x)
        y = s.lin(s.x)
        return (y.detach(), *torch.autograd.grad(y, (s.x,), s.g))
    if kind in ("decode", "layer"):
        s.graph.replay()
        return s.outs
    if kind == "qlora":
        if s.case["dropout"]:
            # the step's random state, as activation checkpointing restores it
            torch.default_generator.manual_seed(s.mask_seed)
        y = qlora_projection(s.x, s.a, s.b, s.packed, s.state, s.bias, SCALING,
                             s.case["dropout"])
        return (y.detach(), *torch.autograd.grad(y, (s.x, s.a, s.b), s.g))
    if kind == "mlp":
        y = fused_qwen2_mlp(s.mlp, s.x)
        return (y.detach(), *torch.autograd.grad(y, (s.x,), s.g))
    if kind == "attention":
        total = sum(s.lengths)
        q, k, v = (t.view(1, total, h, HEAD_DIM).transpose(1, 2)
                   for t, h in zip(s.qkv, s.heads))
        o = packed_causal_attention(q, k, v, s.lengths, HEAD_DIM ** -0.5, cu_seqlens=s.cu)
        return (o.detach(), *torch.autograd.grad(o, s.qkv, s.g))
    if kind == "norm":
        res, y = add_rms_norm(s.r, s.d, s.w, EPS)
        leaves = (s.r, s.d, s.w) if s.case["train_weight"] else (s.r, s.d)
        return (res.detach(), y.detach(), *torch.autograd.grad((res, y), leaves, (s.gs, s.gy)))
    if kind == "head":
        loss, entropy, best, lse = fused_linear_cross_entropy(
            s.x, s.w, s.targets, weight_grad=s.case["weight_grad"])
        mean = loss.sum() / s.labelled
        leaves = (s.x, s.w) if s.case["weight_grad"] else (s.x,)
        return (loss.detach(), entropy, best, lse, *torch.autograd.grad(mean, leaves))
    return dequantize_4bit(s.packed, s.state)


# -------------------------------------------------------------- floor and bounds

def _nf4_bytes(n, k):
    return n * k // 2 + n * k // 64 + n * k // 4096 + 1028


def _pairs(lengths):
    return sum(n * (n + 1) // 2 for n in lengths)


def _add(*parts):
    return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}


def _projection_work(t, n, k, lora, backward):
    """fp16 activations, the NF4 weight read once; LoRA's rank-16 products and tensors."""
    work = {"bytes": _nf4_bytes(n, k) + 2 * t * (n + k), "flops": 2 * t * n * k}
    if lora:
        work["flops"] += 2 * t * RANK * (n + k)
        work["bytes"] += 2 * RANK * (n + k)
    if backward:
        work["flops"] += 2 * t * n * k + (4 * t * RANK * (n + k) if lora else 0)
        work["bytes"] += 2 * t * (n + k) + (2 * RANK * (n + k) if lora else 0)
    return work


def _attention_work(lengths, heads, kv_heads):
    total, pairs = sum(lengths), _pairs(lengths)
    # q, k, v, dO in; o, dq, dk, dv out; two products forward and five backward
    return {"bytes": 2 * total * HEAD_DIM * (4 * heads + 4 * kv_heads),
            "flops": 7 * 2 * HEAD_DIM * pairs * heads}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        return _projection_work(case["t"], case["n"], case["k"], False, case["grad"])
    if kind == "decode":
        t, w = case["t"], [(n, k) for _, n, k in _DECODE]
        return {"bytes": sum(_nf4_bytes(n, k) for n, k in w)
                + 2 * t * (3 * HIDDEN7 + 3 * HIDDEN7 + 2 * KV7),
                "flops": sum(2 * t * n * k for n, k in w)}
    if kind == "qlora":
        return _projection_work(case["t"], case["n"], case["k"], True, True)
    if kind == "mlp":
        t, h, i = case["t"], case["hidden"], case["inter"]
        # x, dY in, Y, dX out; three products forward, three backward
        return {"bytes": 3 * _nf4_bytes(i, h) + 2 * t * 4 * h,
                "flops": 6 * 2 * t * h * i}
    if kind == "attention":
        return _attention_work(_lengths(case), case["heads"], case["kv_heads"])
    if kind == "norm":
        t, h = case["t"], case["h"]
        # r, d, gs, gy in, s, y, dr, dd out; the weight and its gradient
        return {"bytes": 2 * t * h * 8 + 4 * h, "flops": 20 * t * h}
    if kind == "head":
        t = case["t"]
        labelled = 0.635 * t  # rows with a target: the only ones with a gradient
        grads = 2 if case["weight_grad"] else 1
        return {"bytes": 2 * VOCAB * HIDDEN * grads + 2 * t * HIDDEN * 2 + 28 * t,
                "flops": 2 * VOCAB * HIDDEN * (t + grads * labelled)}
    if kind == "dequant":
        return {"bytes": _nf4_bytes(case["n"], case["k"]) + 2 * case["n"] * case["k"],
                "flops": case["n"] * case["k"]}
    lengths = _lengths(case)
    total = sum(lengths)
    parts = [_projection_work(total, n, k, True, True) for _, n, k, _ in _PROJECTIONS]
    work_ = _add(*parts, _attention_work(lengths, HEADS, KV_HEADS))
    # h, dOut in, out, dH out and the weights: what stays if everything between is fused
    work_["bytes"] = 2 * total * HIDDEN * 4 + sum(_nf4_bytes(n, k) + 4 * RANK * (n + k)
                                                  for _, n, k, _ in _PROJECTIONS)
    return work_


def tolerance(case):
    """Four times the error measured against exact() (fp16 results and intermediates, sums
    and softmax in 32 bits): 2.1e-4 to 3.5e-4 for one product, 1.1e-3 for a whole layer."""
    return {
        "linear": {"rel": 1.4e-3},
        "decode": {"rel": 2.6e-3},
        "qlora": {"rel": 1.5e-3},
        "mlp": {"rel": 1.8e-3},
        "attention": {"rel": 1.3e-3},
        "norm": {"rel": 1.7e-3},
        # the first argmax of fp16 logits differs where two of them tie
        "head": {"rel": 1.8e-3, "differ": 0.02},
        "dequant": "exact",
        "layer": {"rel": 4.5e-3},
    }[case["kind"]]


# ------------------------------------------------------------- the same in 64 bits

def _philox_keep(seed, p, rows, cols, dev):
    """The keep mask of the LoRA dropout: word e mod 4 of Philox4x32-10 (Salmon et al.,
    SC'11) at counter e div 4 under the seed, against floor((1 - p) 2^32)."""
    mask = 0xFFFFFFFF

    def mulhilo(m, x):  # 32 x 32 bits in int64 without overflow of the high word
        low, high = (m & 0xFFFF) * x, (m >> 16) * x
        return (high + (low >> 16)) >> 16, ((high << 16) + low) & mask

    n = rows * cols
    g = torch.arange((n + 3) // 4, device=dev, dtype=torch.int64)
    c = [g & mask, g >> 32, torch.zeros_like(g), torch.zeros_like(g)]
    k0, k1 = seed & mask, (seed >> 32) & mask
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
        h0, l0 = mulhilo(0xD2511F53, c[0])
        h1, l1 = mulhilo(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
    p32 = float(torch.tensor(p, dtype=torch.float32))
    keep = torch.stack(c, 1).view(-1)[:n] < int((1.0 - p32) * 4294967296.0)
    return keep.view(rows, cols), 1.0 / (1.0 - p32)


def _attend(q, k, v, g, lengths):
    """Causal attention within each row and its gradients: q, k, v, g [T, heads, 128]."""
    scale, group = HEAD_DIM ** -0.5, q.shape[1] // k.shape[1]
    o, dq = torch.empty_like(q), torch.empty_like(q)
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    start = 0
    for n in lengths:
        rows = slice(start, start + n)
        start += n
        hidden = torch.ones((n, n), dtype=torch.bool, device=q.device).triu(1)
        for h in range(q.shape[1]):
            kv = h // group
            qh, kh, vh, gh = q[rows, h], k[rows, kv], v[rows, kv], g[rows, h]
            p = torch.softmax((qh @ kh.t() * scale).masked_fill(hidden, -math.inf), -1)
            o[rows, h] = p @ vh
            dp = gh @ vh.t()
            ds = p * (dp - (dp * p).sum(-1, keepdim=True)) * scale
            dq[rows, h] = ds @ kh
            dk[rows, kv] += ds.t() @ qh
            dv[rows, kv] += p.t() @ gh
    return o, dq, dk, dv


class _Attend(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, lengths):
        ctx.save_for_backward(q, k, v)
        ctx.lengths = lengths
        return _attend(q, k, v, torch.zeros_like(q), lengths)[0]

    @staticmethod
    def backward(ctx, g):
        return (*_attend(*ctx.saved_tensors, g, ctx.lengths)[1:], None)


def _rms(x, w):
    return w * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), -1) * sin


def _exact_layer(d, lengths):
    f = {name: t.double() for name, t in d.items() if isinstance(t, torch.Tensor)}
    h, total = f["h"].requires_grad_(), sum(lengths)
    leaves = [h]

    def project(name, x):
        p = d[name]
        a, b = p["a"].double().requires_grad_(), p["b"].double().requires_grad_()
        leaves.extend((a, b))
        y = x @ _decoded(p["w"]).double().t() + SCALING * (x @ a.t()) @ b.t()
        return y if p["bias"] is None else y + p["bias"].double()

    cos, sin = f["cos"][0][:, None], f["sin"][0][:, None]
    x = _rms(h, f["norm_in"])
    q = project("q", x).view(total, HEADS, HEAD_DIM)
    k = project("k", x).view(total, KV_HEADS, HEAD_DIM)
    v = project("v", x).view(total, KV_HEADS, HEAD_DIM)
    attn = _Attend.apply(_rotate(q, cos, sin), _rotate(k, cos, sin), v, lengths)
    residual = h + project("o", attn.reshape(total, HIDDEN))
    x = _rms(residual, f["norm_post"])
    act = torch.nn.functional.silu(project("gate", x)) * project("up", x)
    out = residual + project("down", act)
    return (out.detach(), *torch.autograd.grad(out, leaves, f["g"]))


def exact(case, seed):
    kind, d = case["kind"], _inputs(case, seed)
    if kind == "linear":
        w = _decoded(d["w"]).double()
        y = d["x"].double() @ w.t()
        return (y, d["g"].double() @ w) if case["grad"] else y
    if kind == "decode":
        w = {name: _decoded(d[name]).double() for name, _, _ in _DECODE}
        x = d["x_mlp"].double()
        act = torch.nn.functional.silu(x @ w["gate"].t()) * (x @ w["up"].t())
        return (*(d["x"].double() @ w[name].t() for name in ("q", "k", "v")),
                d["x_o"].double() @ w["o"].t(), act @ w["down"].t())
    if kind == "qlora":
        w, x, g = _decoded(d["w"]).double(), d["x"].double(), d["g"].double()
        a, b = d["a"].double(), d["b"].double()
        keep, gain = 1.0, 1.0
        if case["dropout"]:
            gen = torch.Generator().manual_seed(d["mask_seed"])
            seed64 = int(torch.empty((), dtype=torch.int64).random_(generator=gen))
            keep, gain = _philox_keep(seed64, case["dropout"], *x.shape, x.device)
        dropped = x * keep * gain
        y = x @ w.t() + SCALING * (dropped @ a.t()) @ b.t()
        y = y if d["bias"] is None else y + d["bias"].double()
        dz = SCALING * g @ b
        return (y, g @ w + (dz @ a) * keep * gain, dz.t() @ dropped,
                SCALING * g.t() @ (dropped @ a.t()))
    if kind == "mlp":
        w = {name: _decoded(d[name]).double() for name in ("gate", "up", "down")}
        x = d["x"].double().requires_grad_()
        act = torch.nn.functional.silu(x @ w["gate"].t()) * (x @ w["up"].t())
        y = act @ w["down"].t()
        return (y.detach(), *torch.autograd.grad(y, (x,), d["g"].double()))
    if kind == "attention":
        total = sum(_lengths(case))
        q, k, v = (d[name].double().view(total, -1, HEAD_DIM) for name in ("q", "k", "v"))
        o, *grads = _attend(q, k, v, d["g"][0].double(), _lengths(case))
        return (o[None], *(t.reshape(1, total, -1) for t in grads))
    if kind == "norm":
        leaves = [d[name].double().requires_grad_() for name in ("r", "d", "w")]
        res = leaves[0] + leaves[1]
        y = _rms(res, leaves[2])
        wanted = leaves if case["train_weight"] else leaves[:2]
        grads = torch.autograd.grad((res, y), wanted, (d["gs"].double(), d["gy"].double()))
        return (res.detach(), y.detach(), *grads)
    if kind == "head":
        x, w, targets = d["x"].double(), d["w"].double(), d["targets"]
        rows = targets >= 0
        z = x @ w.t()
        lse = torch.logsumexp(z, -1)
        p = z.sub_(lse[:, None])                       # log-probabilities, in place
        picked = p.gather(1, targets.clamp(min=0)[:, None])[:, 0]
        loss = torch.where(rows, -picked, torch.zeros_like(lse))
        entropy = torch.stack([-(r.exp() * r).sum() for r in p])
        p = p.exp_()
        p[torch.arange(len(p), device=p.device), targets.clamp(min=0)] -= 1.0
        p *= (rows / rows.sum())[:, None]
        grads = (p @ w, p.t() @ x) if case["weight_grad"] else (p @ w,)
        return (loss, entropy, None, lse, *grads)
    if kind == "dequant":
        return _decoded(d["w"]).double()
    return _exact_layer(d, _lengths(case))
