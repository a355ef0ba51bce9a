"""Timed cases of the library's main paths, each through a public entry point.

listed() holds fixed cases, draw(rng) gives more of the same ranges;
prepare(case, seed) makes what a program has in hand before the call (inputs,
weights laid out once, a recorded graph), run(state) is one pass, work(case)
its least bytes and operations, tolerance(case) how far another correct
implementation may be off, exact(case, seed) the same outputs in 64 bits by
plain torch.

Kinds of case:
  linear     one Linear: rows x [n, k] weight, bf16, Q8_0 (kept quantised) or fp32
  proj       the q, k, v, gate and up projections of one activation, one launch
  attention  QK-RMSNorm + RoPE on q inside attention over txt | img (bf16), or
             plain fp32 attention
  chain      gated residual + adaLN, then QK-RMSNorm + RoPE with SwiGLU: the
             elementwise work of a single-stream block between its GEMMs
  codec      dequantisation of GGUF weights at load, or their quantisation
  groupnorm  GroupNorm(32) + SiLU of a decoder map
  conv       Conv2d of the decoder, with or without the nearest 2x upscale
  resnet     a decoder ResnetBlock2D through the graph executor
  block      a Flux2 single-stream block through the graph executor
"""
import ctypes
import math
import os
import struct
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "diffusers-cpp_amd"))
import dit_hip as dh  # noqa: E402

HD = 128           # head width
AXES, AXIS = 4, 32  # RoPE axes and their width
EPS = 1e-6
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32, "q8_0": torch.bfloat16}
ES = {"bf16": 2, "f32": 4}
WBYTES = {"bf16": 2.0, "f32": 4.0, "q8_0": 1.125}


# ---------------------------------------------------------------- the cases --
def listed():
    return [
        # The modulation Linear of a double-stream block: one conditioning row,
        # three such products per step.  The smallest call: a weight stream.
        {"name": "modulation_1row_bf16", "kind": "linear", "rows": 1, "n": 18432, "k": 3072, "weights": "bf16"},
        # The text stream's feed-forward output of a double-stream block, with
        # the weights kept as Q8_0 (512 text tokens).
        {"name": "text_down_512_q8", "kind": "linear", "rows": 512, "n": 3072, "k": 9216, "weights": "q8_0"},
        # A single-stream block's input projections for a 33 x 47 image grid
        # and 77 text tokens: ragged rows.
        {"name": "proj_1628_bf16", "kind": "proj", "rows": 1628, "hidden": 3072, "mlp": 9216, "weights": "bf16"},
        # Attention of a 1024 x 1024 image with 512 text tokens.
        {"name": "attention_4608_bf16", "kind": "attention", "dtype": "bf16", "batch": 1, "heads": 24, "txt": 512,
         "gh": 64, "gw": 64},
        # Attention of a 256 x 256 preview with 64 text tokens.
        {"name": "attention_320_bf16", "kind": "attention", "dtype": "bf16", "batch": 1, "heads": 24, "txt": 64,
         "gh": 16, "gw": 16},
        # The elementwise chain of a 1024 x 1024 image.
        {"name": "chain_4608_bf16", "kind": "chain", "dtype": "bf16", "rows": 4608, "heads": 24, "mlp": 9216},
        # Loading a Q4_K feed-forward weight as bf16.
        {"name": "dequant_q4k_3072x9216", "kind": "codec", "what": "dequant", "qtype": "q4_k", "rows": 3072,
         "cols": 9216, "dtype": "bf16"},
        # The norm of a decoder map.
        {"name": "groupnorm_512x256x256_bf16", "kind": "groupnorm", "dtype": "bf16", "n": 1, "c": 512, "h": 256,
         "w": 256},
        # The first upsampling convolution of a 512 px decode tile.
        {"name": "upsample_512x64x64_bf16", "kind": "conv", "dtype": "bf16", "n": 1, "ci": 512, "co": 512, "h": 64,
         "w": 64, "ksize": 3, "up": True},
        # The decoder's last up block of a 512 px tile: its first ResnetBlock2D
        # (256 -> 128 channels, with the 1 x 1 shortcut).
        {"name": "resnet_256to128_512_bf16", "kind": "resnet", "dtype": "bf16", "ci": 256, "co": 128, "h": 512,
         "w": 512},
        # A single-stream block at 512 x 512 (1024 image + 512 text tokens) in
        # the reference's own precision.
        {"name": "block_1536_f32", "kind": "block", "weights": "f32", "txt": 512, "gh": 32, "gw": 32, "heads": 24},
        # A single-stream block at 1024 x 1024 with Q8_0 weights.
        {"name": "block_4608_q8", "kind": "block", "weights": "q8_0", "txt": 512, "gh": 64, "gw": 64, "heads": 24},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "proj", "attention", "attention", "chain", "codec", "groupnorm", "conv",
                       "resnet", "block"])
    if kind == "linear":
        weights = rng.choice(["bf16", "bf16", "q8_0", "f32"])
        k = rng.choice([256, 2560, 3072, 9216, 12288, 64 * rng.randint(2, 144)])
        n = rng.choice([128, 3072, 9216, 18432, _log(rng, 16, 18432)])
        return {"kind": kind, "rows": _log(rng, 1, 1536 if weights == "f32" else 4608), "n": n, "k": k,
                "weights": weights}
    if kind == "proj":
        heads = rng.choice([8, 16, 24])
        return {"kind": kind, "rows": _log(rng, 32, 4608), "hidden": heads * HD, "mlp": 3 * heads * HD,
                "weights": rng.choice(["bf16", "q8_0"])}
    if kind == "attention":
        dtype = rng.choice(["bf16", "bf16", "f32"])
        side = 64 if dtype == "bf16" else 36
        return {"kind": kind, "dtype": dtype, "batch": 1, "heads": rng.choice([2, 8, 16, 24]),
                "txt": rng.randint(1, 512), "gh": rng.randint(4, side), "gw": rng.randint(4, side)}
    if kind == "chain":
        dtype = rng.choice(["bf16", "bf16", "f32"])
        heads = rng.choice([8, 12, 16, 24] if dtype == "bf16" else [4, 8, 12, 16])
        return {"kind": kind, "dtype": dtype, "rows": _log(rng, 16, 4608), "heads": heads, "mlp": 3 * heads * HD}
    if kind == "codec":
        what = rng.choice(["dequant", "dequant", "quantize"])
        qtype = "q8_0" if what == "quantize" else rng.choice(["q8_0", "q4_k"])
        return {"kind": kind, "what": what, "qtype": qtype, "rows": _log(rng, 128, 18432),
                "cols": (32 if qtype == "q8_0" else 256) * (rng.randint(8, 288) if qtype == "q8_0" else
                                                            rng.randint(1, 36)),
                "dtype": "f32" if what == "quantize" else rng.choice(["bf16", "bf16", "f32"])}
    if kind == "groupnorm":
        c = rng.choice([128, 256, 512])
        top = {128: 1024, 256: 700, 512: 512}[c]
        return {"kind": kind, "dtype": rng.choice(["bf16", "f32"]), "n": rng.choice([1, 1, 2]), "c": c,
                "h": _log(rng, 16, top), "w": _log(rng, 16, top)}
    if kind == "conv":
        ci, co = rng.choice([(16, 512), (512, 512), (256, 256), (512, 256), (128, 128), (256, 128), (128, 3)])
        top = {16: 160, 512: 160, 256: 320, 128: 640}[ci]
        ksize = rng.choice([3, 3, 3, 1])
        up = ksize == 3 and ci == co and rng.random() < 0.4
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f32"]), "n": 1, "ci": ci, "co": co,
                "h": _log(rng, 16, top // 2 if up else top), "w": _log(rng, 16, top // 2 if up else top),
                "ksize": ksize, "up": up}
    if kind == "resnet":
        ci, co = rng.choice([(512, 512), (512, 256), (256, 256), (256, 128), (128, 128)])
        top = {512: 160, 256: 320, 128: 640}[ci]
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f32"]), "ci": ci, "co": co,
                "h": _log(rng, 16, top), "w": _log(rng, 16, top)}
    weights = rng.choice(["bf16", "q8_0", "f32"])
    side = 32 if weights == "f32" else 60
    return {"kind": "block", "weights": weights, "txt": rng.randint(1, 512), "gh": rng.randint(8, side),
            "gw": rng.randint(8, side), "heads": rng.choice([8, 16, 24])}


# ------------------------------------------------------------------- inputs --
class _Maker:
    """Seeded inputs on the GPU, the same ones for run and for exact."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def rn(self, shape, dtype=torch.float32, std=1.0, mean=0.0):
        t = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return t.mul_(std).add_(mean).to(dtype)

    def weight(self, n, k, fmt):
        """A Linear weight N(0, 0.02): bf16, fp32, or Q8_0 blocks."""
        if fmt != "q8_0":
            return self.rn((n, k), DTYPES[fmt], 0.02)
        return dh.quantize_q8_0(self.rn((n, k), std=0.02))


def _positions(txt, gh, gw):
    """Text tokens [0, 0, 0, l], then the image grid [0, y, x, 0]."""
    pos = np.zeros((txt + gh * gw, AXES), dtype=np.int32)
    pos[:txt, 3] = np.arange(txt)
    pos[txt:, 1] = np.repeat(np.arange(gh), gw)
    pos[txt:, 2] = np.tile(np.arange(gw), gh)
    return torch.from_numpy(pos).cuda()


def _q8_values(blocks, n, k):
    b = blocks.view(n, k // 32, 34)
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    return (d * b[:, :, 2:].contiguous().view(torch.int8).double()).view(n, k)


def _weight64(w, n, k, fmt):
    """The values a Linear multiplies by: Q8_0 weights are their bf16-rounded block values."""
    return _q8_values(w, n, k).bfloat16().double() if fmt == "q8_0" else w.double()


def _linear_inputs(c, seed):
    m = _Maker(seed)
    x = m.rn((c["rows"], c["k"]), DTYPES[c["weights"]])
    return x, m.weight(c["n"], c["k"], c["weights"])


def _proj_widths(c):
    return [c["hidden"]] * 3 + [c["mlp"]] * 2


def _proj_inputs(c, seed):
    m = _Maker(seed)
    x = m.rn((c["rows"], c["hidden"]), torch.bfloat16)
    return x, [m.weight(n, c["hidden"], c["weights"]) for n in _proj_widths(c)]


def _attention_inputs(c, seed):
    m = _Maker(seed)
    dt, S = DTYPES[c["dtype"]], c["txt"] + c["gh"] * c["gw"]
    q = m.rn((c["batch"], S, c["heads"], HD), dt)
    k = m.rn((c["batch"], S, c["heads"], HD), dt)
    v = m.rn((c["batch"], S, c["heads"], HD), dt)
    return q, k, v, m.rn((HD,), std=0.02, mean=1.0), m.rn((HD,), std=0.02, mean=1.0)


def _chain_inputs(c, seed):
    m = _Maker(seed)
    dt, S, D = DTYPES[c["dtype"]], c["rows"], c["heads"] * HD
    t = {"h": m.rn((S, D), dt), "o": m.rn((S, D), dt), "q": m.rn((S, c["heads"], HD), dt),
         "k": m.rn((S, c["heads"], HD), dt), "gu": m.rn((S, 2 * c["mlp"]), dt)}
    for v in ("gate", "shift", "scale"):
        t[v] = m.rn((D,), std=0.1)
    t["wq"], t["wk"] = m.rn((HD,), std=0.02, mean=1.0), m.rn((HD,), std=0.02, mean=1.0)
    side = max(1, int(math.sqrt(S - S // 9)))
    t["pos"] = torch.cat([_positions(S - side * side, 1, 0), _positions(0, side, side)])
    return t


def _q4k_blocks(m, rows, cols):
    """Q4_K super-blocks (fp16 d, dmin; packed 6-bit scales; 4-bit codes) with trained-weight magnitudes."""
    nb = rows * cols // 256
    b = torch.randint(0, 256, (nb, 144), generator=m.g, device="cuda", dtype=torch.uint8)
    b[:, 0:2] = (m.rn((nb,), std=1e-4).abs() + 1e-5).half().view(torch.uint8).view(nb, 2)
    b[:, 2:4] = (m.rn((nb,), std=1e-4).abs() + 1e-5).half().view(torch.uint8).view(nb, 2)
    return b.view(-1)


def _codec_inputs(c, seed):
    m = _Maker(seed)
    if c["qtype"] == "q4_k":
        return _q4k_blocks(m, c["rows"], c["cols"])
    w = m.rn((c["rows"], c["cols"]), std=0.02)
    return w if c["what"] == "quantize" else dh.quantize_q8_0(w).view(-1)


def _groupnorm_inputs(c, seed):
    m = _Maker(seed)
    return (m.rn((c["n"], c["c"], c["h"], c["w"]), DTYPES[c["dtype"]]), m.rn((c["c"],), std=0.02, mean=1.0),
            m.rn((c["c"],), std=0.02))


def _conv_weight(m, co, ci, k):
    return m.rn((co, ci, k, k), std=1.0 / math.sqrt(ci * k * k)), m.rn((co,), std=0.1)


def _conv_inputs(c, seed):
    m = _Maker(seed)
    return (m.rn((c["n"], c["ci"], c["h"], c["w"]), DTYPES[c["dtype"]]),) + _conv_weight(m, c["co"], c["ci"], c["ksize"])


def _resnet_inputs(c, seed):
    m = _Maker(seed)
    t = {"x": m.rn((1, c["ci"], c["h"], c["w"]), DTYPES[c["dtype"]])}
    for i, (a, b) in ((1, (c["co"], c["ci"])), (2, (c["co"], c["co"]))):
        t["gw%d" % i], t["gb%d" % i] = m.rn((b,), std=0.02, mean=1.0), m.rn((b,), std=0.02)
        t["w%d" % i], t["b%d" % i] = _conv_weight(m, a, b, 3)
    if c["ci"] != c["co"]:
        t["ws"], t["bs"] = _conv_weight(m, c["co"], c["ci"], 1)
    return t


BLOCK_WEIGHTS = (("q", 1, 1), ("k", 1, 1), ("v", 1, 1), ("gate", 3, 1), ("up", 3, 1), ("out", 1, 1), ("down", 1, 3))


def _block_inputs(c, seed):
    """x, the modulation vector, norm weights, and the seven Linear weights (out, in)."""
    m = _Maker(seed)
    S, D = c["txt"] + c["gh"] * c["gw"], c["heads"] * HD
    t = {"x": m.rn((1, S, D), DTYPES[c["weights"]]), "mod": m.rn((1, 1, 3 * D), std=0.1),
         "wq": m.rn((HD,), std=0.02, mean=1.0), "wk": m.rn((HD,), std=0.02, mean=1.0)}
    for name, n, k in BLOCK_WEIGHTS:
        t["W" + name] = m.weight(n * D, k * D, c["weights"])
    return t


# -------------------------------------------------------------------- graphs --
def _fbits(v):
    return struct.unpack("<i", struct.pack("<f", v))[0]


_BACKEND = None


def _backend():
    """One backend per process, as a program keeps it."""
    global _BACKEND
    if _BACKEND is None:
        h = ctypes.c_void_p()
        dh.check(dh.load().dt_backend_init(0, ctypes.byref(h)), "dt_backend_init")
        _BACKEND = h
    dh.check(dh.load().dt_backend_set_stream(_BACKEND, dh.stream()), "dt_backend_set_stream")
    return _BACKEND


class _Graph:
    """A recorded ggml-shaped graph; ne in ggml order, every node with memory of its own."""

    TORCH = {dh.F32: torch.float32, dh.BF16: torch.bfloat16, dh.I32: torch.int32}

    def __init__(self):
        self.nodes, self.keep = [], []

    def leaf(self, t):
        self.keep.append(t)
        return dh.desc(t)

    def new(self, op, ne, type_, srcs, params=()):
        t = torch.empty([int(n) for n in reversed(ne)], dtype=self.TORCH[type_], device="cuda")
        d = dh.desc(t, op)
        self.keep.append(t)
        return self._record(d, srcs, params)

    def _record(self, d, srcs, params):
        for i, s in enumerate(srcs):
            d.src[i] = ctypes.pointer(s)
        for i, p in enumerate(params):
            d.op_params[i] = p
        self.nodes.append(d)
        return d

    def view(self, src, ne, nb, off=0):
        d = dh.DtTensor()
        d.type, d.op, d.data = src.type, dh.OP_VIEW, (src.data or 0) + off
        for i in range(4):
            d.ne[i], d.nb[i] = ne[i], nb[i]
        return self._record(d, [src], [off])

    def reshape(self, src, ne):
        ne = list(ne) + [1] * (4 - len(ne))
        nb = [src.nb[0]]
        for i in range(3):
            nb.append(nb[-1] * ne[i])
        return self.view(src, ne, nb)

    def swap12(self, x):
        ne, nb = x.ne, x.nb
        return self.view(x, [ne[0], ne[2], ne[1], ne[3]], [nb[0], nb[2], nb[1], nb[3]])

    def binary(self, op, a, b):
        return self.new(op, list(a.ne), a.type, [a, b])

    def silu(self, a):
        return self.binary(dh.OP_MUL, a, self.new(dh.OP_SIGMOID, list(a.ne), a.type, [a]))

    def mul_mat(self, w, x):
        return self.new(dh.OP_MUL_MAT, [w.ne[1], x.ne[1], x.ne[2], x.ne[3]], x.type, [w, x])

    def ready(self, out):
        out.flags |= dh.FLAG_OUTPUT
        self.array = (ctypes.POINTER(dh.DtTensor) * len(self.nodes))(*[ctypes.pointer(d) for d in self.nodes])
        self.out = next(t for t in self.keep if t.data_ptr() == out.data)
        return self

    def compute(self, backend):
        dh.check(dh.load().dt_graph_compute(backend, self.array, len(self.nodes)), "dt_graph_compute")
        return self.out


def _weight_leaf(g, w, n, k, fmt):
    if fmt != "q8_0":
        return g.leaf(w)
    lib = dh.load()
    buf = torch.empty(lib.dt_q8_0_split_bytes(n, k), dtype=torch.uint8, device="cuda")
    scales = buf.data_ptr() + lib.dt_q8_0_split_scale_offset(n, k)
    dh.check(lib.dt_q8_0_split(ctypes.c_void_p(w.data_ptr()), n, k, k // 32 * 34, ctypes.c_void_p(buf.data_ptr()), k,
                               ctypes.c_void_p(scales), n, dh.stream()), "dt_q8_0_split")
    g.keep.append(buf)
    d = dh.DtTensor()
    d.type, d.data = 100, buf.data_ptr()  # DT_TYPE_Q8_0_SPLIT
    for i, (ne, nb) in enumerate(((k, 1), (n, k), (1, n * k), (1, n * k))):
        d.ne[i], d.nb[i] = ne, nb
    return d


def _block_graph(c, t):
    """Flux2SingleTransformerBlock::forward, node for node."""
    g = _Graph()
    S, H = c["txt"] + c["gh"] * c["gw"], c["heads"]
    D = H * HD
    x, mod = g.leaf(t["x"]), g.leaf(t["mod"])
    es = x.nb[0]
    W = {n: _weight_leaf(g, t["W" + n], a * D, b * D, c["weights"]) for n, a, b in BLOCK_WEIGHTS}
    part = [g.view(mod, [D, 1, 1, 1], [4, 12 * D, 12 * D, 12 * D], 4 * D * i) for i in range(3)]
    one = g.new(dh.OP_FILL, [1, 1, 1, 1], dh.F32, [], [_fbits(1.0)])
    t1 = g.binary(dh.OP_ADD, part[1], one)
    n = g.new(dh.OP_NORM, list(x.ne), x.type, [x], [_fbits(EPS)])
    y = g.binary(dh.OP_ADD, g.binary(dh.OP_MUL, n, t1), part[0])
    p = {a: g.mul_mat(W[a], y) for a in ("q", "k", "v", "gate", "up")}
    posn = g.leaf(_positions(c["txt"], c["gh"], c["gw"]))
    cols = []
    for a in range(AXES):
        v = g.view(posn, [1, S, 1, 1], [4, 16, 16 * S, 16 * S], 4 * a)
        cols.append(g.reshape(g.new(dh.OP_CPY, [1, S, 1, 1], dh.I32, [v]), [S]))

    def heads(z):
        return g.reshape(z, [HD, H, S])

    def qk(z, w):
        r = g.new(dh.OP_RMS_NORM, [HD, H, S, 1], z.type, [heads(z)], [_fbits(EPS)])
        return g.binary(dh.OP_MUL, r, g.leaf(w))

    def rope(z):
        out = None
        for a, col in enumerate(cols):
            v = g.view(z, [AXIS, H, S, 1], list(z.nb), a * AXIS * es)
            r = g.new(dh.OP_ROPE, [AXIS, H, S, 1], z.type, [v, col],
                      [AXIS, 0, _fbits(2000.0), _fbits(1.0), _fbits(0.0), _fbits(1.0)])
            out = r if out is None else g.new(dh.OP_CONCAT, [out.ne[0] + AXIS, H, S, 1], z.type, [out, r], [0])
        return out

    q, k = qk(p["q"], t["wq"]), qk(p["k"], t["wk"])
    q, k = rope(q), rope(k)
    at = g.new(dh.OP_FLASH_ATTN_EXT, [HD, H, S, 1], x.type, [g.swap12(q), g.swap12(k), g.swap12(heads(p["v"]))],
               [_fbits(1.0 / math.sqrt(HD))])
    mlp = g.binary(dh.OP_MUL, g.silu(p["gate"]), p["up"])
    o = g.binary(dh.OP_ADD, g.mul_mat(W["out"], g.reshape(at, [D, S])), g.mul_mat(W["down"], mlp))
    return g.ready(g.binary(dh.OP_ADD, x, g.binary(dh.OP_MUL, o, part[2])))


def _resnet_graph(c, t):
    """ResnetBlock2D::forward (no temb), node for node, conv weights packed at load."""
    g = _Graph()

    def vec(v):
        return g.reshape(g.leaf(v), [1, 1, v.numel()])

    def norm(z, w, b):
        Wd, Hd, C, N = list(z.ne)
        v = g.reshape(z, [Wd * Hd * C // 32, 32, N])
        v = g.reshape(g.new(dh.OP_NORM, list(v.ne), z.type, [v], [_fbits(EPS)]), [Wd, Hd, C, N])
        return g.silu(g.binary(dh.OP_ADD, g.binary(dh.OP_MUL, v, vec(w)), vec(b)))

    def conv(z, w, b):
        co, ci, k, _ = w.shape
        pk = dh.conv2d_pack(w)
        g.keep.append(pk.packed)
        d = dh.DtTensor()
        d.type, d.data = 101, pk.packed.data_ptr()  # DT_TYPE_CONV2D_PACKED
        for i, ne in enumerate((k, k, ci, co)):
            d.ne[i], d.nb[i] = ne, 1
        y = g.new(dh.OP_CONV_2D_DIRECT, [z.ne[0], z.ne[1], co, z.ne[3]], z.type, [d, z], [1, 1, k // 2, k // 2, 1, 1])
        return g.binary(dh.OP_ADD, y, vec(b))

    x = g.leaf(t["x"])
    h = conv(norm(x, t["gw1"], t["gb1"]), t["w1"], t["b1"])
    h = conv(norm(h, t["gw2"], t["gb2"]), t["w2"], t["b2"])
    s = conv(x, t["ws"], t["bs"]) if "ws" in t else x
    y = g.binary(dh.OP_ADD, s, h)
    return g.ready(g.new(dh.OP_SCALE, list(y.ne), y.type, [y], [_fbits(1.0)]))


# ------------------------------------------------------------- prepare, run --
def prepare(case, seed):
    c = case
    k = c["kind"]
    s = {"case": c}
    if k == "linear":
        s["x"], w = _linear_inputs(c, seed)
        s["w"] = dh.q8_0_split(w, c["n"], c["k"]) if c["weights"] == "q8_0" else w
    elif k == "proj":
        s["x"], ws = _proj_inputs(c, seed)
        s["w"] = [dh.q8_0_split(w, n, c["hidden"]) if c["weights"] == "q8_0" else w for w, n in zip(ws, _proj_widths(c))]
    elif k == "attention":
        s["q"], s["k"], s["v"], s["w0"], s["w1"] = _attention_inputs(c, seed)
        s["pos"] = _positions(c["txt"], c["gh"], c["gw"])
        s["table"] = dh.rope_table(512, AXIS, 2000.0)
    elif k == "chain":
        s.update(_chain_inputs(c, seed))
        s["table"] = dh.rope_table(512, AXIS, 10000.0)
    elif k == "codec":
        s["src"] = _codec_inputs(c, seed)
    elif k == "groupnorm":
        s["x"], s["gw"], s["gb"] = _groupnorm_inputs(c, seed)
    elif k == "conv":
        s["x"], w, s["b"] = _conv_inputs(c, seed)
        s["w"] = dh.conv2d_pack(w)
    elif k == "resnet":
        s["backend"], s["graph"] = _backend(), _resnet_graph(c, _resnet_inputs(c, seed))
    elif k == "block":
        s["backend"], s["graph"] = _backend(), _block_graph(c, _block_inputs(c, seed))
    return s


def run(state):
    s, c = state, state["case"]
    k = c["kind"]
    if k == "linear":
        return {"q8_0": dh.gemm_q8_0, "bf16": dh.gemm, "f32": dh.gemm_f32}[c["weights"]](s["x"], s["w"])
    if k == "proj":
        outs = [torch.empty((c["rows"], n), dtype=torch.bfloat16, device="cuda") for n in _proj_widths(c)]
        return dh.gemm_grouped([(s["x"], w, o) for w, o in zip(s["w"], outs)])
    if k == "attention":
        if c["dtype"] == "f32":
            return dh.flash_attn_f32(s["q"], s["k"], s["v"])
        q, T = s["q"], c["txt"]
        return dh.flash_attn_qk([(q[:, :T], s["w0"]), (q[:, T:], s["w1"])], s["k"], s["v"], s["pos"], AXIS, 2000.0,
                                EPS, table=s["table"])
    if k == "chain":
        r, y = dh.gated_residual_adaln(s["h"], s["o"], s["gate"], s["shift"], s["scale"], EPS)
        I = c["mlp"]
        q, kk, m = dh.qk_rmsnorm_rope_swiglu(s["q"], s["k"], s["wq"], s["wk"], s["pos"], AXIS, 10000.0,
                                             s["gu"][:, :I], s["gu"][:, I:], EPS, table=s["table"])
        return {"r": r, "y": y, "q": q, "k": kk, "mlp": m}
    if k == "codec":
        if c["what"] == "quantize":
            return dh.quantize_q8_0(s["src"])
        return dh.dequant(s["src"], dh.Q8_0 if c["qtype"] == "q8_0" else dh.Q4_K, c["rows"], c["cols"],
                          DTYPES[c["dtype"]])
    if k == "groupnorm":
        return dh.groupnorm_silu(s["x"], 32, s["gw"], s["gb"], EPS)
    if k == "conv":
        return dh.conv2d(s["x"], s["w"], s["b"], upscale2=c["up"])
    return s["graph"].compute(s["backend"])


# ------------------------------------------------------------ work, tolerance --
def work(case):
    c = case
    k = c["kind"]
    if k == "linear":
        act = ES["f32" if c["weights"] == "f32" else "bf16"]
        return {"bytes": act * c["rows"] * (c["k"] + c["n"]) + WBYTES[c["weights"]] * c["n"] * c["k"],
                "flops": 2.0 * c["rows"] * c["n"] * c["k"]}
    if k == "proj":
        n = sum(_proj_widths(c))
        return {"bytes": 2 * c["rows"] * (c["hidden"] + n) + WBYTES[c["weights"]] * n * c["hidden"],
                "flops": 2.0 * c["rows"] * n * c["hidden"]}
    if k == "attention":
        S = c["txt"] + c["gh"] * c["gw"]
        return {"bytes": 4.0 * ES[c["dtype"]] * c["batch"] * S * c["heads"] * HD,
                "flops": 4.0 * c["batch"] * c["heads"] * S * S * HD}
    if k == "chain":
        return {"bytes": ES[c["dtype"]] * c["rows"] * (8.0 * c["heads"] * HD + 3 * c["mlp"]) + 16 * c["rows"],
                "flops": 0}
    if k == "codec":
        n = float(c["rows"] * c["cols"])
        packed = 34 / 32 if c["qtype"] == "q8_0" else 144 / 256
        return {"bytes": n * (packed + ES[c["dtype"]]), "flops": 0}
    if k == "groupnorm":
        return {"bytes": 2.0 * ES[c["dtype"]] * c["n"] * c["c"] * c["h"] * c["w"], "flops": 0}
    if k == "conv":
        px, f = c["n"] * c["h"] * c["w"], 4 if c["up"] else 1
        taps = c["ci"] * c["co"] * c["ksize"] ** 2
        return {"bytes": ES[c["dtype"]] * px * (c["ci"] + f * c["co"]) + 2.0 * taps, "flops": 2.0 * f * px * taps}
    if k == "resnet":
        px = c["h"] * c["w"]
        taps = 9 * c["co"] * (c["ci"] + c["co"]) + (c["ci"] * c["co"] if c["ci"] != c["co"] else 0)
        return {"bytes": ES[c["dtype"]] * px * (c["ci"] + c["co"]) + 2.0 * taps, "flops": 2.0 * px * taps}
    S, D = c["txt"] + c["gh"] * c["gw"], c["heads"] * HD
    act = ES["f32" if c["weights"] == "f32" else "bf16"]
    return {"bytes": 2.0 * act * S * D + WBYTES[c["weights"]] * 13 * D * D, "flops": 26.0 * S * D * D + 4.0 * S * S * D}


def tolerance(case):
    """About four times the relative error against exact() that was measured over each kind's sizes."""
    k = case["kind"]
    if k == "codec":
        return "exact"
    half = case.get("weights", case.get("dtype")) != "f32"
    if k == "conv":
        return {"rel": 9.5e-3}  # operands rounded to bf16 in either type
    if k == "resnet":
        return {"rel": 1.4e-2}
    if k == "attention":
        return {"rel": 1.2e-2 if half else 1.2e-6}
    if k == "linear":
        return {"rel": 7e-3 if half else 1e-6}
    if k == "block":
        return {"rel": 7.2e-3 if half else 2.4e-7}
    return {"rel": 7e-3 if half else 4e-7}


# ---------------------------------------------------------------------- exact --
def _rope_angles(pos, base):
    """[S, 64] angles: theta_0 = p, theta_{i + 1} = theta_i * base^(-2/32) in fp32 per axis (ggml's rule)."""
    step = np.float32(np.power(np.float32(base), np.float32(-2.0 / AXIS)))
    p = pos.cpu().numpy().astype(np.float32)
    cols = []
    for a in range(AXES):
        th = p[:, a].copy()
        for _ in range(AXIS // 2):
            cols.append(th.astype(np.float64))
            th = (th * step).astype(np.float32)
    return torch.from_numpy(np.stack(cols, 1)).cuda()


def _qk64(q, w, pos, base):
    """RMSNorm over the head, weights, rotation of adjacent pairs; q [S, H, 128] in 64 bits."""
    z = q * torch.rsqrt(q.square().mean(-1, keepdim=True) + EPS) * w.double()
    th = _rope_angles(pos, base)[:, None, :]
    a, b = z[..., 0::2], z[..., 1::2]
    return torch.stack([a * th.cos() - b * th.sin(), a * th.sin() + b * th.cos()], -1).reshape(q.shape)


def _attn64(q, k, v):
    """q, k, v [S, H, 128] in 64 bits, head by head."""
    o = torch.empty_like(q)
    for h in range(q.shape[1]):
        p = torch.softmax(q[:, h] @ k[:, h].t() / math.sqrt(HD), -1)
        o[:, h] = p @ v[:, h]
    return o


def _conv64(x, w, b):
    """[1, Ci, H, W] by [Co, Ci, K, K] with padding K // 2, tap by tap, in 64 bits."""
    n, ci, H, W = x.shape
    K = w.shape[2]
    y = b.double().view(1, -1, 1, 1).expand(n, w.shape[0], H, W).clone()
    xp = torch.nn.functional.pad(x, [K // 2] * 4)
    for i in range(K):
        for j in range(K):
            for m in range(n):
                y[m] += (w[:, :, i, j].double() @ xp[m, :, i:i + H, j:j + W].reshape(ci, -1)).view(-1, H, W)
    return y


def _gn64(x, w, b):
    n, C = x.shape[:2]
    v = x.reshape(n, 32, -1)
    v = (v - v.mean(-1, keepdim=True)) * torch.rsqrt(v.var(-1, unbiased=False, keepdim=True) + EPS)
    return torch.nn.functional.silu(v.view(x.shape) * w.double().view(1, C, 1, 1) + b.double().view(1, C, 1, 1))


def _ln64(x):
    return (x - x.mean(-1, keepdim=True)) * torch.rsqrt(x.var(-1, unbiased=False, keepdim=True) + EPS)


def _q4k64(b, rows, cols):
    b = b.view(-1, 144)
    d = b[:, 0:2].contiguous().view(torch.float16).double()
    dm = b[:, 2:4].contiguous().view(torch.float16).double()
    s = b[:, 4:16].long()
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    qs = b[:, 16:].view(-1, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
    return ((d * sc)[:, :, None] * q - (dm * mn)[:, :, None]).view(rows, cols)


def exact(case, seed):
    c = case
    k = c["kind"]
    if k == "linear":
        x, w = _linear_inputs(c, seed)
        return x.double() @ _weight64(w, c["n"], c["k"], c["weights"]).t()
    if k == "proj":
        x, ws = _proj_inputs(c, seed)
        return [x.double() @ _weight64(w, n, c["hidden"], c["weights"]).t() for w, n in zip(ws, _proj_widths(c))]
    if k == "attention":
        q, kk, v, w0, w1 = _attention_inputs(c, seed)
        q, kk, v = q.double(), kk.double(), v.double()
        if c["dtype"] != "f32":
            T, pos = c["txt"], _positions(c["txt"], c["gh"], c["gw"])
            q = torch.cat([torch.cat([_qk64(z[:T], w0, pos[:T], 2000.0), _qk64(z[T:], w1, pos[T:], 2000.0)])[None]
                           for z in q])
        return torch.stack([_attn64(q[b], kk[b], v[b]) for b in range(c["batch"])])
    if k == "chain":
        t = _chain_inputs(c, seed)
        r = t["h"].double() + t["gate"].double() * t["o"].double()
        gate, up = t["gu"][:, :c["mlp"]].double(), t["gu"][:, c["mlp"]:].double()
        return {"r": r, "y": (1 + t["scale"].double()) * _ln64(r.to(t["h"].dtype).double()) + t["shift"].double(),
                "q": _qk64(t["q"].double(), t["wq"], t["pos"], 10000.0),
                "k": _qk64(t["k"].double(), t["wk"], t["pos"], 10000.0), "mlp": torch.nn.functional.silu(gate) * up}
    if k == "codec":
        if c["what"] == "quantize":
            return None
        b = _codec_inputs(c, seed)
        return (_q8_values if c["qtype"] == "q8_0" else _q4k64)(b, c["rows"], c["cols"])
    if k == "groupnorm":
        x, w, b = _groupnorm_inputs(c, seed)
        return _gn64(x.double(), w, b)
    if k == "conv":
        x, w, b = _conv_inputs(c, seed)
        x = x.double()
        if c["up"]:
            x = x.repeat_interleave(2, 2).repeat_interleave(2, 3)
        return _conv64(x, w, b)
    if k == "resnet":
        t = _resnet_inputs(c, seed)
        x = t["x"].double()
        h = _conv64(_gn64(x, t["gw1"], t["gb1"]), t["w1"], t["b1"])
        h = _conv64(_gn64(h, t["gw2"], t["gb2"]), t["w2"], t["b2"])
        return (_conv64(x, t["ws"], t["bs"]) if "ws" in t else x) + h
    t = _block_inputs(c, seed)
    S, D, H = c["txt"] + c["gh"] * c["gw"], c["heads"] * HD, c["heads"]
    W = {n: _weight64(t["W" + n], a * D, b * D, c["weights"]).t() for n, a, b in BLOCK_WEIGHTS}
    shift, scale, gate = t["mod"].double().view(3, D)
    x = t["x"].double()[0]
    y = _ln64(x) * (1 + scale) + shift
    pos = _positions(c["txt"], c["gh"], c["gw"])
    q = _qk64((y @ W["q"]).view(S, H, HD), t["wq"], pos, 2000.0)
    kk = _qk64((y @ W["k"]).view(S, H, HD), t["wk"], pos, 2000.0)
    at = _attn64(q, kk, (y @ W["v"]).view(S, H, HD)).view(S, D)
    mlp = torch.nn.functional.silu(y @ W["gate"]) * (y @ W["up"])
    return (x + gate * (at @ W["out"] + mlp @ W["down"])).view(1, S, D)
