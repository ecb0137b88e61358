"""What the speed of this package is measured on: encoder passes through
execution plans, quantized matrix products and block decoding, with inputs
made from a seed alone and 64-bit results in plain torch.

Weights are N(0, 0.02) quantized here to the GGUF block formats, token ids
are uniform with BOS first, norm weights N(1, 0.1). Encoder passes either run
all 16 layers or four of them (one before the token merge, three after it: the
same share as 4 of 16) at the full model's widths.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PACKAGE = os.path.join(_ROOT, "nemotron-3-embed-webgpu_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

HIDDEN, VOCAB, KV_HEADS, EPS, THETA = 2048, 131072, 8, 1e-5, 1e6
KV_THRESHOLD, KV_STRIDE = 2048, 3
# query heads, head dim, FFN width
SHAPES = {"benchmark": (32, 64, 8192), "published": (24, 128, 6144)}
TYPES = {"q4_0": 2, "q4_k": 12, "q6_k": 14}
BLOCK = {"q4_0": (32, 18), "q4_k": (256, 144), "q6_k": (256, 210)}  # values, bytes


def _encode(name, shape, layers, lengths, host):
    c = {"path": "encode", "shape": shape, "layers": layers, "lengths": ",".join(map(str, lengths)), "host": host}
    return dict(c, name=name) if name else c


def _matmul(name, kind, m, n, k):
    c = {"path": "matmul", "type": kind, "m": m, "n": n, "k": k}
    return dict(c, name=name) if name else c


def _dequant(name, kind, values, out):
    c = {"path": "dequant", "type": kind, "values": values, "out": out}
    return dict(c, name=name) if name else c


RAGGED = [15, 15, 50, 50, 150, 150, 500, 500, 15, 50, 150, 500, 15, 50, 150, 500]


def listed():
    return [
        # one short query, whole model: what an interactive search waits for
        _encode("encode_1x15", "benchmark", 16, [15], False),
        # 16 concurrent requests of 150 tokens, whole model: the benchmark's headline
        _encode("encode_16x150", "benchmark", 16, [150] * 16, False),
        # one passage through the host call at the published model's widths and pack storage
        _encode("layers_1x150_host", "published", 4, [150], True),
        # one page of text
        _encode("layers_1x500", "benchmark", 4, [500], False),
        # a micro-batch of queries and passages of mixed lengths
        _encode("layers_ragged16", "benchmark", 4, RAGGED, False),
        # one long document: sampled keys in the attention
        _encode("layers_1x5000", "benchmark", 4, [5000], False),
        # indexing long passages in full batches: the most tokens in one pass
        _encode("layers_8x1500", "published", 4, [1500] * 8, False),
        # gate/up for one short query
        _matmul("matmul_15_q4k", "q4_k", 15, 16384, 2048),
        # the down projection for a passage of 96 merged tokens
        _matmul("matmul_96_q6k", "q6_k", 96, 2048, 8192),
        # the published model's gate/up projection for a page, a ragged row count
        _matmul("matmul_333_q40", "q4_0", 333, 12288, 2048),
        # gate/up for 16 x 150 tokens, the benchmark's dominant product
        _matmul("matmul_2400_q4k", "q4_k", 2400, 16384, 2048),
        # decoding a model's worth of blocks
        _dequant("dequant_q4k_f16", "q4_k", 302 * 10**6 // 144 * 256, "f16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    top = max((work(c)["flops"] for c in listed()))
    while True:
        path = rng.choice(["encode", "encode", "matmul", "dequant"])
        if path == "encode":
            batch = rng.choice([1, 1, 2, 3, 5, 8, 13, 16])
            longest = _log_int(rng, 1, 5000)
            # requests of one length, or of any up to the longest
            lengths = [longest] * batch if rng.random() < 0.4 else [_log_int(rng, 1, longest) for _ in range(batch)]
            c = _encode(None, rng.choice(sorted(SHAPES)), 4, lengths, rng.random() < 0.3)
        elif path == "matmul":
            n = _log_int(rng, 256, 16384)
            n = n if rng.random() < 0.2 else max(128, n // 128 * 128)
            c = _matmul(None, rng.choice(sorted(TYPES)), _log_int(rng, 1, 4096), n, 256 * rng.choice([4, 6, 8, 12, 24, 32]))
        else:
            c = _dequant(None, rng.choice(sorted(TYPES)), 256 * _log_int(rng, 4096, 2 * 10**6), rng.choice(["f16", "f32"]))
        # padded tokens of a plan stay within the largest listed pass too
        if path == "encode" and max(lengths) * len(lengths) > 12000:
            continue
        if work(c)["flops"] <= top:
            return c


# ---- inputs ------------------------------------------------------------------


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _half_bytes(t):
    return t.half().contiguous().view(torch.uint8).reshape(*t.shape, 2)


def _quantize(kind, w):
    """GGUF blocks (uint8 [blocks, bytes]) of the values `w` (float32, whole blocks)."""
    if kind == "q4_0":
        v = w.reshape(-1, 32)
        top = v.gather(1, v.abs().argmax(1, keepdim=True))
        d = (top / -8).half()
        inv = torch.where(d == 0, torch.zeros_like(top), 1 / d.float())
        q = (v * inv + 8.5).floor().clamp(0, 15).to(torch.uint8)
        return torch.cat([_half_bytes(d)[:, 0], q[:, :16] | (q[:, 16:] << 4)], 1)
    if kind == "q4_k":
        v = w.reshape(-1, 8, 32)
        low = (-v.amin(2)).clamp(min=0)
        step = (v.amax(2) + low) / 15
        d, dmin = (step.amax(1, keepdim=True) / 63).half(), (low.amax(1, keepdim=True) / 63).half()
        sc = (step / d.float()).round().clamp(1, 63)
        mn = (low / dmin.float()).round().clamp(0, 63)
        q = ((v + (dmin.float() * mn)[..., None]) / (d.float() * sc)[..., None]).round().clamp(0, 15).to(torch.uint8)
        sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
        scales = torch.cat([(sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6), (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6),
                            (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
        nibbles = q[:, 0::2] | (q[:, 1::2] << 4)
        return torch.cat([_half_bytes(d)[:, 0], _half_bytes(dmin)[:, 0], scales, nibbles.reshape(-1, 128)], 1)
    v = w.reshape(-1, 16, 16)
    step = v.abs().amax(2) / 31
    d = (step.amax(1, keepdim=True) / 127).half()
    sc = (step / d.float()).round().clamp(1, 127)
    q = ((v / (d.float() * sc)[..., None]).round().clamp(-32, 31) + 32).to(torch.uint8)
    q = q.reshape(-1, 2, 4, 32)  # [block][half][quadrant][lane]
    ql = (q[:, :, :2] & 15) | ((q[:, :, 2:] & 15) << 4)
    qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
    return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.uint8), _half_bytes(d)[:, 0]], 1)


def _matrix(g, kind, n, k):
    """Blocks of an n x k matrix of N(0, 0.02) weights."""
    return _quantize(kind, torch.randn(n * k, device="cuda", generator=g) * 0.02)


def _widths(case):
    heads, hd, ffn = SHAPES[case["shape"]]
    return heads, hd, ffn, (heads + 2 * KV_HEADS) * hd, heads * hd


def _layers(case, g):
    """Per layer: norm weights and the blocks of the four matrices. The
    benchmark's storage is Q4_K with a Q6_K down projection, the published
    pack's Q4_0 throughout."""
    heads, hd, ffn, qkv, qw = _widths(case)
    bench = case["shape"] == "benchmark"
    kind, down = ("q4_k", "q6_k") if bench else ("q4_0", "q4_0")
    for _ in range(case["layers"]):
        yield {"attn_norm": 1 + 0.1 * torch.randn(HIDDEN, device="cuda", generator=g),
               "ffn_norm": 1 + 0.1 * torch.randn(HIDDEN, device="cuda", generator=g),
               "attn_qkv": (kind, qkv, HIDDEN, _matrix(g, kind, qkv, HIDDEN)),
               "attn_output": (kind, HIDDEN, qw, _matrix(g, kind, HIDDEN, qw)),
               "ffn_gate_up": (kind, 2 * ffn, HIDDEN, _matrix(g, kind, 2 * ffn, HIDDEN)),
               "ffn_down": (down, HIDDEN, ffn, _matrix(g, down, HIDDEN, ffn))}


def _lengths(case):
    return [int(v) for v in case["lengths"].split(",")]


def _ids(case, g):
    lengths = _lengths(case)
    ids = torch.randint(1, VOCAB, (len(lengths), max(lengths)), device="cuda", generator=g, dtype=torch.int32)
    ids[:, 0] = 1
    for b, n in enumerate(lengths):
        ids[b, n:] = 0
    return ids


def _table(g):
    return (torch.randn(VOCAB, HIDDEN, device="cuda", generator=g) * 0.02).half()


def _merge_after(case):
    return case["layers"] // 4


_streams = []


def _stream():
    """One stream for the whole program, as a server has: passes follow each other."""
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0]


class _Encoder:
    """A model, its plan and the buffers of one program; given back with it."""

    def __init__(self, case, seed):
        from nemo_amd import runtime as rt
        g = _generator(seed)
        heads, hd, ffn, _, _ = _widths(case)
        self.lengths = np.array(_lengths(case), dtype=np.uint32)
        self.ids = _ids(case, g)
        out_norm = 1 + 0.1 * torch.randn(HIDDEN, device="cuda", generator=g)
        source = {"token_embd.weight": (rt.TYPE_F16, [HIDDEN, VOCAB], _table(g).cpu().numpy()),
                  "output_norm.weight": (rt.TYPE_F32, [HIDDEN], out_norm.cpu().numpy())}
        for i, layer in enumerate(_layers(case, g)):
            for name, v in layer.items():
                key = "blk.%d.%s.weight" % (i, name)
                if isinstance(v, tuple):
                    kind, n, k, blocks = v
                    source[key] = (TYPES[kind], [k, n], blocks.cpu().numpy())
                else:
                    source[key] = (rt.TYPE_F32, [HIDDEN], v.cpu().numpy())
        dims = rt.make_dims(q_heads=heads, head_dim=hd, intermediate=ffn, layers=case["layers"],
                            merge_after_layer=_merge_after(case))
        self.model = rt.NemotronHipModel(source, dims=dims)
        self.plan = self.model.createPlan(len(self.lengths), int(self.lengths.max()))
        self.out = torch.empty(len(self.lengths), HIDDEN, device="cuda")
        self.host_ids = self.ids.cpu().numpy().view(np.uint32).reshape(-1) if case["host"] else None
        self.stream = _stream().cuda_stream

    def run(self):
        if self.host_ids is not None:
            return self.plan.run_sync(self.host_ids, self.lengths)
        self.plan.run_device(self.ids.data_ptr(), self.lengths, self.out.data_ptr(), self.stream)
        return self.out

    def __del__(self):
        for held in ("plan", "model"):
            if hasattr(self, held):
                getattr(self, held).destroy()


class _Product:
    """Y = X W^T with a weight on the device."""

    def __init__(self, case, seed):
        from nemo_amd import runtime as rt
        self.m = case["m"]
        self.x, blocks = _product_inputs(case, seed)
        self.w = rt.QuantWeight(TYPES[case["type"]], case["n"], case["k"], blocks.cpu().numpy())
        self.y = torch.empty(self.m, case["n"], dtype=torch.float16, device="cuda")
        self.stream = _stream().cuda_stream

    def run(self):
        self.w.matmul(self.x.data_ptr(), self.m, self.y.data_ptr(), stream=self.stream)
        return self.y


class _Decode:
    """Raw blocks on the device to values."""

    def __init__(self, case, seed):
        from nemo_amd import runtime as rt
        self.call = rt.dequantize_device
        self.type, self.values = TYPES[case["type"]], case["values"]
        self.raw = _decode_inputs(case, seed)
        self.half = case["out"] == "f16"
        self.out = torch.empty(self.values, dtype=torch.float16 if self.half else torch.float32, device="cuda")
        self.stream = _stream().cuda_stream

    def run(self):
        p = self.out.data_ptr()
        self.call(self.type, self.raw.data_ptr(), self.values, 0 if self.half else p, p if self.half else 0, self.stream)
        return self.out


def _product_inputs(case, seed):
    g = _generator(seed)
    x = torch.randn(case["m"], case["k"], device="cuda", generator=g).half()
    return x, _matrix(g, case["type"], case["n"], case["k"])


def _decode_inputs(case, seed):
    # whole 64 MB runs of weights at a time: the float32 values need not all be held
    g = _generator(seed)
    values, step = case["values"], 1 << 26
    return torch.cat([_quantize(case["type"], torch.randn(min(step, values - i), device="cuda", generator=g) * 0.02)
                      for i in range(0, values, step)])


def prepare(case, seed):
    state = {"encode": _Encoder, "matmul": _Product, "dequant": _Decode}[case["path"]](case, seed)
    torch.cuda.synchronize()  # inputs are made on another stream than the passes run on
    return state


def run(state):
    return state.run()


# ---- what a pass cannot do without --------------------------------------------


def _merged(n):
    return max(1, math.ceil(n * 0.64))


def _keys(n):
    s = KV_STRIDE if n > KV_THRESHOLD else 1
    return (n + s - 1) // s


def work(case):
    if case["path"] == "encode":
        heads, hd, ffn, qkv, qw = _widths(case)
        lengths = _lengths(case)
        weights = HIDDEN * qkv + qw * HIDDEN + 3 * HIDDEN * ffn
        flops = 0
        for i in range(case["layers"]):
            rows = lengths if i < _merge_after(case) else [_merged(n) for n in lengths]
            flops += 2 * weights * sum(rows) + sum(4 * qw * n * _keys(n) for n in rows)
        if case["shape"] == "benchmark":
            matrices = (weights - HIDDEN * ffn) * 144 / 256 + HIDDEN * ffn * 210 / 256
        else:
            matrices = weights * 18 / 32
        tokens = sum(lengths)
        return {"bytes": case["layers"] * (matrices + 8 * HIDDEN) + tokens * (4 + 2 * HIDDEN) + 4 * HIDDEN * len(lengths),
                "flops": flops}
    per, size = BLOCK[case["type"]]
    if case["path"] == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": n * k // per * size + 2 * m * (n + k), "flops": 2 * m * n * k}
    return {"bytes": case["values"] // per * size + case["values"] * (2 if case["out"] == "f16" else 4),
            "flops": 2 * case["values"]}


def tolerance(case):
    if case["path"] == "dequant":
        return "exact"
    if case["path"] == "matmul":
        # f16 weights, activations and results with sums in 32 bits (2.9e-4
        # and 1.3e-3 from the 64-bit product)
        return {"rel": 1.2e-3, "max": 5e-3}
    # f16 activations between the operations of 16 or 4 layers (up to 2.2e-3
    # and 1.6e-3 from 64 bits, the most for the fewest tokens)
    return {"rel": 9e-3 if case["layers"] > 4 else 6e-3}


# ---- the same in 64 bits --------------------------------------------------------


def _decode(kind, blocks):
    """float64 values of GGUF blocks (uint8 [blocks, bytes]), in order."""
    def half(a):
        return blocks[:, a:a + 2].contiguous().view(torch.float16).double()

    if kind == "q4_0":
        q = blocks[:, 2:]
        return (half(0) * (torch.cat([q & 15, q >> 4], 1).double() - 8)).reshape(-1)
    if kind == "q4_k":
        s = blocks[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        b = blocks[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([b & 15, b >> 4], 2).reshape(-1, 8, 32).double()
        return ((half(0) * sc)[..., None] * q - (half(2) * mn)[..., None]).reshape(-1)
    ql, qh = blocks[:, :128].reshape(-1, 2, 2, 32), blocks[:, 128:192].reshape(-1, 2, 32)
    low = torch.cat([ql & 15, ql >> 4], 2)
    high = torch.stack([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
    q = (low | (high << 4)).reshape(-1, 16, 16).double() - 32
    sc = blocks[:, 192:208].contiguous().view(torch.int8).double()
    return ((half(208) * sc)[..., None] * q).reshape(-1)


def _weights(matrix):
    kind, n, k, blocks = matrix
    return _decode(kind, blocks).reshape(n, k)


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w.double()


def _rotation(n, hd):
    """cos and sin of the YaRN-scaled rotary angles, [n][hd / 2]."""
    pairs = hd // 2
    bound = lambda beta: hd * math.log(16384.0 / (beta * 2 * math.pi)) / (2 * math.log(THETA))  # noqa: E731
    lo, hi = math.floor(bound(32)), math.ceil(bound(1))
    i = torch.arange(pairs, dtype=torch.float64, device="cuda")
    ramp = 1 - ((i - lo) / max(0.001, hi - lo)).clamp(0, 1)
    angle = torch.arange(n, dtype=torch.float64, device="cuda")[:, None] * THETA ** (-i / pairs) * ((1 - ramp) / 16 + ramp)
    return angle.cos(), angle.sin()


def _rotate(x, cos, sin):  # [heads][n][hd], pairs adjacent
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack([e * cos - o * sin, e * sin + o * cos], -1).flatten(-2)


def _attention(qkv, heads, hd):
    n = qkv.shape[0]
    cos, sin = _rotation(n, hd)
    q, k, v = (t.reshape(n, -1, hd).transpose(0, 1) for t in qkv.split([heads * hd, KV_HEADS * hd, KV_HEADS * hd], 1))
    s = KV_STRIDE if n > KV_THRESHOLD else 1
    q, k, v = _rotate(q, cos, sin), _rotate(k, cos, sin)[:, ::s], v[:, ::s]
    group = heads // KV_HEADS
    out = [torch.softmax(q[h] @ k[h // group].T.contiguous() / math.sqrt(hd), 1) @ v[h // group] for h in range(heads)]
    return torch.stack(out, 1).reshape(n, heads * hd)


def _merge(x):
    """The first row, then the means of adjacent rows, 64 % of them in all."""
    n, t = x.shape[0], _merged(x.shape[0])
    rows = [x[0]]
    for p in range(1, t):
        start = 1 + (p - 1) * (n - 1) // (t - 1)
        end = min(n, max(1 + p * (n - 1) // (t - 1), start + 1))
        rows.append(x[start:end].mean(0))
    return torch.stack(rows)


def exact(case, seed):
    if case["path"] == "dequant":
        blocks = _decode_inputs(case, seed)
        out = torch.cat([_decode(case["type"], b).float() for b in blocks.split(1 << 18)])
        return out.half() if case["out"] == "f16" else out
    if case["path"] == "matmul":
        x, blocks = _product_inputs(case, seed)
        return x.double() @ _weights((case["type"], case["n"], case["k"], blocks)).T
    g = _generator(seed)
    heads, hd, ffn, _, _ = _widths(case)
    lengths = _lengths(case)
    ids = _ids(case, g)
    out_norm = 1 + 0.1 * torch.randn(HIDDEN, device="cuda", generator=g)
    table = _table(g)
    rows = list(lengths)
    x = torch.cat([table[ids[b, :n].long()] for b, n in enumerate(lengths)]).double()
    layers = list(_layers(case, g))
    normed = _norm(x, layers[0]["attn_norm"])
    for i, layer in enumerate(layers):
        if i == _merge_after(case):
            x = torch.cat([_merge(part) for part in x.split(rows)])
            normed = torch.cat([_merge(part) for part in normed.split(rows)])
            rows = [_merged(n) for n in rows]
        qkv = normed @ _weights(layer["attn_qkv"]).T
        att = torch.cat([_attention(part, heads, hd) for part in qkv.split(rows)])
        x = x + att @ _weights(layer["attn_output"]).T
        gate, up = (_norm(x, layer["ffn_norm"]) @ _weights(layer["ffn_gate_up"]).T).split(ffn, 1)
        x = x + (gate * torch.sigmoid(gate) * up) @ _weights(layer["ffn_down"]).T
        normed = _norm(x, layers[i + 1]["attn_norm"] if i + 1 < len(layers) else out_norm)
    mean = torch.stack([part.mean(0) for part in normed.split(rows)])
    mean = mean / mean.norm(dim=1, keepdim=True)
    return list(mean) if case["host"] else mean
