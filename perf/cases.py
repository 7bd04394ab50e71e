"""What this library is used for, as timed cases: the quantized operators a model runtime calls, over the range of sizes
such a runtime meets, and the decode loop of a small int4 language model.

Five kinds of work, each through the package's public entry points:

  linear4   MatMulNBits on a prepacked weight: rows from one (a decode step) to thousands (a prompt)
  ffn8      a dynamically quantized feed-forward block: DynamicQuantizeLinear, MatMulInteger with the fused rescale,
            GELU or ReLU, DynamicQuantizeLinear, MatMulInteger
  dense8    a statically quantized dense layer: QLinearMatMul
  conv8     a statically quantized convolution: QLinearConv, along one axis (vocoders, speech encoders) or two (vision)
  decode    tokens of a gemma3-1b-shaped decoder from a filled cache, one replayed graph per token

``listed()`` are the cases that are always timed, ``draw()`` gives others of the same ranges.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from __graft_entry__ import load_package

pkg = load_package()
ops, dec = pkg.ops, pkg.decoder

_DEVICE = "cuda:0"
_ctx = None


def _context():
    """One context per process, as a runtime keeps it."""
    global _ctx
    if _ctx is None:
        _ctx = pkg.Context(0)
    return _ctx


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # one activation row, one projection (gate and up side by side): the call a decode loop makes
        dict(name="linear4_row", kind="linear4", rows=1, k=1152, n=13824, block=32, zp=True, dtype="f32", level=0),
        # a few sequences decoded together: the down projection (long k, few columns) ...
        dict(name="linear4_rows8_down", kind="linear4", rows=8, k=6912, n=1152, block=32, zp=True, dtype="f32", level=0),
        # ... and the unembedding, whose weight is read once per step
        dict(name="linear4_rows4_unembed", kind="linear4", rows=4, k=1152, n=262144, block=32, zp=True, dtype="f32", level=0),
        # a prompt in half precision, symmetric weights with large blocks
        dict(name="linear4_prompt_f16", kind="linear4", rows=512, k=2048, n=11008, block=128, zp=False, dtype="f16", level=0),
        # a prompt of no particular length in single precision, the element type exported graphs carry
        dict(name="linear4_prompt_f32", kind="linear4", rows=333, k=1152, n=13824, block=32, zp=True, dtype="f32", level=0),
        # a dynamically quantized encoder block over ten seconds of speech frames ...
        dict(name="ffn8_1000", kind="ffn8", tokens=1000, d=1024, f=4096, act="gelu"),
        # ... and over one short chunk of a stream
        dict(name="ffn8_chunk", kind="ffn8", tokens=23, d=1024, f=4096, act="relu"),
        # a large statically quantized layer
        dict(name="dense8_4096", kind="dense8", rows=4096, k=4096, n=4096, per_column=True),
        # a dilated convolution along time, as vocoders stack them
        dict(name="conv8_time", kind="conv8", batch=1, c_in=192, c_out=192, h=1, w=4096, kh=1, kw=7, stride=1, dil=3, group=1),
        # a 3 x 3 convolution of an image classifier, a batch of images
        dict(name="conv8_image", kind="conv8", batch=8, c_in=128, c_out=128, h=28, w=28, kh=3, kw=3, stride=1, dil=1, group=1),
        # eight greedy tokens behind a context of 2048, every layer global
        dict(name="decode_2048", kind="decode", context=2048, local_layers=False, tokens=8),
        # the same behind a long context, five of six layers seeing their last 512 positions only
        dict(name="decode_long", kind="decode", context=8000, local_layers=True, tokens=8),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(v, of):
    return max(of, (v + of // 2) // of * of)


def draw(rng):
    kind = rng.choices(["linear4", "ffn8", "dense8", "conv8", "decode"], [9, 3, 3, 4, 1])[0]
    if kind == "linear4":
        dtype = rng.choice(["f32", "f16"])
        case = dict(kind=kind, rows=_log_uniform(rng, 1, 2048), k=_multiple(_log_uniform(rng, 512, 11008), 32),
                    n=_log_uniform(rng, 512, 16384), block=rng.choice([32, 32, 32, 64, 128, 128, 16, 256]), zp=rng.random() < 0.6,
                    dtype=dtype, level=rng.choice([0, 4]) if dtype == "f32" else 0)
        if rng.random() < 0.8:              # projections are whole multiples of a head's width; gathered vocabularies are not
            case["n"] = _multiple(case["n"], 64)
        # what one pass may cost; blocks of 16 are met in small models
        case["rows"] = max(1, min(case["rows"], int((2e10 if case["block"] == 16 else 1.3e11) / (2 * case["k"] * case["n"]))))
        if case["rows"] <= 8 and rng.random() < 0.15:
            case["n"], case["k"] = _log_uniform(rng, 32768, 262144), _multiple(_log_uniform(rng, 512, 1152), 32)
        return case
    if kind == "ffn8":
        d = _multiple(_log_uniform(rng, 256, 2048), 64)
        return dict(kind=kind, tokens=_log_uniform(rng, 1, 4096), d=d, f=d * rng.choice([2, 4]), act=rng.choice(["gelu", "relu"]))
    if kind == "dense8":
        return dict(kind=kind, rows=_log_uniform(rng, 1, 4096), k=_log_uniform(rng, 128, 4096) if rng.random() < 0.2 else _multiple(_log_uniform(rng, 128, 4096), 64),
                    n=_log_uniform(rng, 128, 4096) if rng.random() < 0.3 else _multiple(_log_uniform(rng, 128, 4096), 64), per_column=rng.random() < 0.7)
    if kind == "conv8":
        form = rng.choices(["time", "image", "point", "depth", "stem"], [4, 4, 2, 1, 1])[0]
        if form == "time":
            c = _multiple(_log_uniform(rng, 32, 512), 16)
            return dict(kind=kind, batch=_log_uniform(rng, 1, 8), c_in=c, c_out=c, h=1, w=_log_uniform(rng, 256, 8192), kh=1,
                        kw=rng.choice([3, 5, 7, 11]), stride=rng.choice([1, 1, 1, 2]), dil=rng.choice([1, 3, 5]), group=1)
        side, batch = _log_uniform(rng, 7, 112), _log_uniform(rng, 1, 16)
        c = min(512, _multiple(int(4096 / side * rng.choice([0.5, 1, 1.5])), 16))     # deep layers are small and wide
        if form == "image":
            return dict(kind=kind, batch=batch, c_in=c, c_out=c * rng.choice([1, 1, 2]), h=side, w=side, kh=3, kw=3,
                        stride=rng.choice([1, 1, 2]), dil=1, group=1)
        if form == "point":
            return dict(kind=kind, batch=batch, c_in=c, c_out=c * rng.choice([1, 4]), h=side, w=side, kh=1, kw=1, stride=1, dil=1, group=1)
        if form == "depth":
            return dict(kind=kind, batch=batch, c_in=c, c_out=c, h=side, w=side, kh=3, kw=3, stride=rng.choice([1, 2]), dil=1, group=c)
        return dict(kind=kind, batch=batch, c_in=3, c_out=_multiple(rng.randint(24, 72), 8), h=224, w=224, kh=7, kw=7, stride=2, dil=1, group=1)
    return dict(kind=kind, context=_log_uniform(rng, 16, 8000), local_layers=rng.random() < 0.5, tokens=rng.randint(2, 8))


# ------------------------------------------------------------------- operands

def _generator(seed):
    return torch.Generator(device=_DEVICE).manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=_DEVICE)


def _uniform(g, lo, hi, *shape):
    return lo + (hi - lo) * torch.rand(*shape, generator=g, device=_DEVICE)


def _bytes(g, lo, hi, *shape, dtype=torch.uint8):
    """Whole numbers lo..hi."""
    return torch.randint(lo, hi + 1, shape, generator=g, device=_DEVICE, dtype=torch.int32).to(dtype)


def _host(t):
    return t.cpu().numpy()


def _nbits(g, k, n, block, zp=True, scale=1.0):
    """A random int4 weight in the operator's layout, as a model file holds it: (B, scales, zero points or None)."""
    blocks = -(-k // block)
    B = _host(_bytes(g, 0, 255, n, blocks, block // 2))
    scales = _host(_uniform(g, 0.005, 0.05, n * blocks) * scale)
    return B, scales, _host(_bytes(g, 0, 255, n, (blocks + 1) // 2)) if zp else None


class _State:
    """What a program keeps between calls; gives the library's handles back when it goes."""

    def __init__(self, case):
        self.ctx = _context()
        self.kind = case["kind"]
        self.handles, self.graph, self.decoder = [], None, None

    def keep(self, handle):
        self.handles.append(handle)
        return handle

    def __del__(self):
        self.ctx.flush()
        if self.graph is not None:
            self.ctx.graph_destroy(self.graph)
        if self.decoder is not None:
            self.decoder.destroy()
        for h in self.handles:
            h.destroy()
        self.ctx.flush()


def prepare(case, seed):
    g = _generator(seed)
    s = _State(case)
    globals()["_prepare_" + case["kind"]](case, g, s)
    torch.cuda.synchronize()
    return s


def run(state):
    return globals()["_run_" + state.kind](state)


# -------------------------------------------------------------------- linear4

def _prepare_linear4(c, g, s):
    B, scales, zp = _nbits(g, c["k"], c["n"], c["block"], c["zp"], 0.5 * math.sqrt(1152 / c["k"]))
    f16 = c["dtype"] == "f16"
    dt = torch.float16 if f16 else torch.float32
    s.weight = s.keep(ops.NBitsWeight(s.ctx, B, scales.astype(np.float16) if f16 else scales, zp, c["k"], c["n"], c["block"]))
    s.x = _normal(g, c["rows"], c["k"]).to(dt)
    s.y = torch.empty(c["rows"], c["n"], dtype=dt, device=_DEVICE)
    s.dtype, s.rows, s.level = pkg.F16 if f16 else pkg.F32, c["rows"], c["level"]


def _run_linear4(s):
    ops.matmul_nbits_packed_device(s.ctx, s.x.data_ptr(), s.dtype, s.weight, s.y.data_ptr(), s.rows, s.level)
    return s.y


# ----------------------------------------------------------------------- ffn8

def _prepare_ffn8(c, g, s):
    t, d, f = c["tokens"], c["d"], c["f"]
    s.t, s.d, s.f, s.act = t, d, f, c["act"]
    s.w1 = s.keep(ops.Int8Weight(s.ctx, _host(_bytes(g, -127, 127, d, f, dtype=torch.int8))))
    s.w2 = s.keep(ops.Int8Weight(s.ctx, _host(_bytes(g, -127, 127, f, d, dtype=torch.int8))))
    # weight scales that keep every row's products near 1
    s.s1 = _uniform(g, 0.5, 1.5, f) / (73.0 * math.sqrt(d))
    s.s2 = _uniform(g, 0.5, 1.5, d) / (73.0 * math.sqrt(f))
    s.b1, s.b2 = 0.1 * _normal(g, f), 0.1 * _normal(g, d)
    s.x = _normal(g, t, d)
    s.xq = torch.empty(t, d, dtype=torch.uint8, device=_DEVICE)
    s.h = torch.empty(t, f, device=_DEVICE)
    s.hq = torch.empty(t, f, dtype=torch.uint8, device=_DEVICE)
    s.y = torch.empty(t, d, device=_DEVICE)
    # each quantizer's scale (4 bytes), zero point (1 byte) and, behind a ReLU, the range slot its producer fills
    s.q = torch.zeros(32, dtype=torch.uint8, device=_DEVICE)


def _run_ffn8(s):
    ctx, q = s.ctx, s.q.data_ptr()
    sx, zx, sh, zh, slot = q, q + 4, q + 8, q + 12, q + 16
    ops.dynamic_quantize_linear_device(ctx, s.x.data_ptr(), s.t * s.d, s.xq.data_ptr(), sx, zx)
    if s.act == "relu":
        ctx.fill(slot, 0, 8, 0)
        ops.matmul_integer_scale_bias_device(ctx, s.xq.data_ptr(), pkg.U8, s.w1, zx, None, sx, 0, s.s1.data_ptr(), 1,
                                             s.b1.data_ptr(), 1, True, slot, s.h.data_ptr(), s.t)
        ops.dynamic_quantize_linear_device(ctx, s.h.data_ptr(), s.t * s.f, s.hq.data_ptr(), sh, zh, slot, True)
    else:
        ops.matmul_integer_scale_bias_device(ctx, s.xq.data_ptr(), pkg.U8, s.w1, zx, None, sx, 0, s.s1.data_ptr(), 1,
                                             s.b1.data_ptr(), 1, False, None, s.h.data_ptr(), s.t)
        ctx._check(ctx.lib.hipc_dynamic_quantize_linear_gelu(ctx.handle, s.h.data_ptr(), s.t * s.f, ops.SQRT2_F32, 1.0, 0.5, 0,
                                                             s.hq.data_ptr(), sh, zh, None))
    ops.matmul_integer_scale_bias_device(ctx, s.hq.data_ptr(), pkg.U8, s.w2, zh, None, sh, 0, s.s2.data_ptr(), 1,
                                         s.b2.data_ptr(), 1, False, None, s.y.data_ptr(), s.t)
    return s.y


# --------------------------------------------------------------------- dense8

def _prepare_dense8(c, g, s):
    m, k, n = c["rows"], c["k"], c["n"]
    s.weight = s.keep(ops.Int8Weight(s.ctx, _host(_bytes(g, -127, 127, k, n, dtype=torch.int8))))
    s.w_scale = _host(_uniform(g, 0.5, 1.5, n if c["per_column"] else 1) * 0.01)
    s.x = _bytes(g, 0, 255, m, k)
    s.y = torch.empty(m, n, dtype=torch.uint8, device=_DEVICE)
    s.rows = m
    s.y_scale = 0.02 * 0.01 * 74.0 * 73.0 * math.sqrt(k) / 40.0      # one standard deviation is some 40 codes


def _run_dense8(s):
    ops.qlinear_matmul_device(s.ctx, s.x.data_ptr(), pkg.U8, 0.02, 128, s.weight, s.w_scale, 0, s.y_scale, 128, pkg.U8,
                              s.y.data_ptr(), s.rows)
    return s.y


# ---------------------------------------------------------------------- conv8

def _conv_pads(c):
    return c["dil"] * (c["kh"] - 1) // 2, c["dil"] * (c["kw"] - 1) // 2


def _conv_out(c):
    ph, pw = _conv_pads(c)
    return ((c["h"] + 2 * ph - c["dil"] * (c["kh"] - 1) - 1) // c["stride"] + 1,
            (c["w"] + 2 * pw - c["dil"] * (c["kw"] - 1) - 1) // c["stride"] + 1)


def _prepare_conv8(c, g, s):
    ph, pw = _conv_pads(c)
    x_shape = (c["batch"], c["c_in"], c["h"], c["w"])
    w_shape = (c["c_out"], c["c_in"] // c["group"], c["kh"], c["kw"])
    sh = 1 if c["h"] == 1 else c["stride"]
    s.geom = pkg.ConvGeom.make(x_shape, w_shape, (sh, c["stride"]), (1 if c["h"] == 1 else c["dil"], c["dil"]), (ph, pw, ph, pw), c["group"])
    s.weight = s.keep(ops.ConvWeight(s.ctx, _host(_bytes(g, -127, 127, *w_shape, dtype=torch.int8)), s.geom))
    s.w_scale = _host(_uniform(g, 0.5, 1.5, c["c_out"]) * 0.01)
    s.x = _bytes(g, 0, 255, *x_shape)
    s.bias = _bytes(g, -4096, 4096, c["c_out"], dtype=torch.int32)
    s.y = torch.empty(ops.conv_out_shape(s.ctx, s.geom), dtype=torch.uint8, device=_DEVICE)
    k = w_shape[1] * c["kh"] * c["kw"]
    s.y_scale = 0.02 * 0.01 * 74.0 * 73.0 * math.sqrt(k) / 40.0


def _run_conv8(s):
    ops.qlinear_conv_device(s.ctx, s.x.data_ptr(), pkg.U8, 0.02, 128, s.weight, s.w_scale, 0, s.y_scale, 128, pkg.U8,
                            s.bias.data_ptr(), s.geom, s.y.data_ptr())
    return s.y


# --------------------------------------------------------------------- decode

def _prepare_decode(c, g, s):
    cfg, ctx = dict(dec.GEMMA3_1B), s.ctx
    qd, kvd = cfg["n_q_heads"] * cfg["head_dim"], cfg["n_kv_heads"] * cfg["head_dim"]
    shapes = {dec.QKV: (cfg["hidden"], qd + 2 * kvd), dec.O: (qd, cfg["hidden"]), dec.GATE_UP: (cfg["hidden"], 2 * cfg["ffn"]),
              dec.DOWN: (cfg["ffn"], cfg["hidden"])}

    def near_one(n):
        return _host(1.0 + 0.1 * _normal(g, n))

    w = dec.Weights(cfg)
    for layer in range(cfg["n_layers"]):
        for which, (k, n) in shapes.items():
            w.linears[(layer, which)] = _nbits(g, k, n, cfg["block_size"], True, 0.5 * math.sqrt(1152 / k))
        for which in (dec.NORM_INPUT, dec.NORM_POST_ATTN, dec.NORM_PRE_FFN, dec.NORM_POST_FFN):
            w.norms[(layer, which)] = near_one(cfg["hidden"])
        for which in (dec.NORM_Q, dec.NORM_K):
            w.norms[(layer, which)] = near_one(cfg["head_dim"])
    w.linears[(0, dec.LM_HEAD)] = _nbits(g, cfg["hidden"], cfg["vocab"], cfg["block_size"], True, 0.5)
    w.norms[(0, dec.NORM_FINAL)] = near_one(cfg["hidden"])
    w.embedding = _nbits(g, cfg["hidden"], cfg["vocab"], cfg["block_size"])

    d = s.decoder = dec.Decoder(ctx, cfg, c["context"] + 64)
    d.load(w)
    rows = (cfg["n_kv_heads"], c["context"], cfg["head_dim"])
    for layer in range(cfg["n_layers"]):
        if c["local_layers"] and layer % 6 != 5:
            d.set_layer_attention(layer, 512, 10000.0)
        elif c["local_layers"]:
            d.set_layer_attention(layer, 0, 1e6)
        d.fill_cache(layer, _host(_normal(g, *rows).half()), _host(_normal(g, *rows).half()))
    s.context, s.tokens, s.first = c["context"], c["tokens"], int(_bytes(g, 0, cfg["vocab"] - 1, 1, dtype=torch.int32))
    # one step as it is, one recorded
    d.reset(s.first, s.context)
    d.step()
    ctx.flush()
    ctx.capture_begin()
    d.step()
    s.graph = ctx.capture_end()


def _run_decode(s):
    s.decoder.reset(s.first, s.context)
    for _ in range(s.tokens):
        s.ctx.graph_launch(s.graph)
    _, _, logits, history = s.decoder.read(want_logits=True, n_history=s.context + s.tokens)
    return logits, history[s.context:]       # the history before the context is not this run's


# ----------------------------------------------------------- work and tolerance

def work(case):
    c = case
    if c["kind"] == "linear4":
        blocks, size = -(-c["k"] // c["block"]), 2 if c["dtype"] == "f16" else 4
        weight = c["n"] * (blocks * (c["block"] // 2 + size) + ((blocks + 1) // 2 if c["zp"] else 0))
        return {"bytes": weight + c["rows"] * (c["k"] + c["n"]) * size, "flops": 2 * c["rows"] * c["k"] * c["n"]}
    if c["kind"] == "ffn8":
        t, d, f = c["tokens"], c["d"], c["f"]
        # every operator's tensors: x f32 -> codes; codes -> h f32; h -> codes; codes -> y f32; both weights
        return {"bytes": t * (5 * d + d + 4 * f + 5 * f + f + 4 * d) + 2 * d * f + 8 * (d + f), "flops": 4 * t * d * f}
    if c["kind"] == "dense8":
        m, k, n = c["rows"], c["k"], c["n"]
        return {"bytes": m * k + k * n + m * n, "flops": 2 * m * k * n}
    if c["kind"] == "conv8":
        ho, wo = _conv_out(c)
        taps, outs = c["c_in"] // c["group"] * c["kh"] * c["kw"], c["batch"] * c["c_out"] * ho * wo
        return {"bytes": c["batch"] * c["c_in"] * c["h"] * c["w"] + c["c_out"] * (taps + 8) + outs, "flops": 2 * outs * taps}
    cfg = dec.GEMMA3_1B
    kv = 2 * 2 * cfg["n_kv_heads"] * cfg["head_dim"]         # bytes of one position in one layer
    weights = dec.bytes_per_token(cfg, 0)
    n_local = sum(1 for layer in range(cfg["n_layers"]) if layer % 6 != 5) if c["local_layers"] else 0
    seen = n_local * min(512, c["context"]) + (cfg["n_layers"] - n_local) * c["context"]
    matrix = (cfg["n_layers"] * (1152 * 1536 + 1024 * 1152 + 1152 * 13824 + 6912 * 1152) + 1152 * cfg["vocab"]) * 2
    return {"bytes": c["tokens"] * (weights + kv * seen), "flops": c["tokens"] * (matrix + 4 * cfg["n_q_heads"] * cfg["head_dim"] * seen)}


def tolerance(case):
    if case["kind"] == "linear4":
        if case["dtype"] == "f16" or case["level"] >= 2:
            return {"rel": 5e-4}         # f16 results, or activations of 11 bits (accuracy_level 2 and above allows them)
        return {"rel": 1e-5}             # f32 sums over k
    if case["kind"] == "ffn8" and case["act"] == "gelu":
        # erf's exponential differs in its last bits between implementations, and a value next to a tie of the quantizer
        # then takes the neighbouring code
        return {"rel": 3e-4, "max": 1e-2}
    if case["kind"] == "decode":
        # keys and values are kept in f16: a last-bit difference of a sum moves some of them by half a unit of 11 bits
        return {"rel": 1e-3, "max": 2e-2}
    return "exact"                       # whole numbers, and float results with every rounding defined
