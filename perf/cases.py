"""Representative workloads of the GGUF quantized-linear path, and how to time and check one.

A case is the linears that a program runs between its other kernels, through ``tensor_amd.torch``:
kernels are loaded once, calls on fixed buffers are prepared once (``Kernel.prepare``; bound calls of
the provider for the dequantizer), and a pass submits them in order on PyTorch's current stream.  Kinds (``op``):

* ``layer``: the seven linears of ``layers`` decoder layers (q, k, v, o, gate, up, down; hidden
  size ``hidden``, k and v rows ``kv``, MLP size ``ffn``) on ``m`` activation rows.  ``down`` is
  the encoding of the down projection, ``encoding`` that of the other six.  ``entry`` is how the
  program calls them: ``linear`` is one ``gguf_linear`` per matrix; ``group`` shares launches
  (m <= 8: grouped GEMV for q + k + v, the SwiGLU pair for gate and up; above: grouped GEMM with
  its workspace).  Every linear has activations of its own, so that each output stands for itself.
* ``head``: one wide ``gguf_linear`` with fp32 logits.
* ``packed``: one call of the shape-fixed packed form, fp32 activations and output.
* ``dequant``: ``count`` weight matrices to ``out`` elements.

Several layers (or matrices) make a pass's weights larger than the caches, as a model's are.
"""

from __future__ import annotations

import functools
import math

import torch

import tensor_amd.torch as tt
from tensor_amd.torch.session import session

# encoding: (elements per block, bytes per block)
GEOMETRY = {"q4_0": (32, 18), "q4_1": (32, 20), "q5_0": (32, 22), "q5_1": (32, 24), "q8_0": (32, 34),
            "q2_k": (256, 84), "q3_k": (256, 110), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210)}
GEMV_ROWS = 8  # rows the decode entries take; above, a program calls the grouped GEMM


def _layer(name, entry, encoding, down, hidden, kv, ffn, m, layers):
    return {"name": name, "op": "layer", "entry": entry, "encoding": encoding, "down": down, "hidden": hidden,
            "kv": kv, "ffn": ffn, "m": m, "layers": layers}


def listed():
    return [
        # the showcase's single call: the smallest work a program submits, bound by latency
        {"name": "packed_m1_q4_k_1024", "op": "packed", "encoding": "q4_k", "m": 1, "n": 1024, "k": 1024},
        # one token of an 8B-class model in the usual mix (Q4_K, Q6_K down), launches shared
        _layer("decode_m1_q4_k_4096", "group", "q4_k", "q6_k", 4096, 1024, 12288, 1, 2),
        # its vocabulary projection
        {"name": "head_m1_q6_k_151936", "op": "head", "encoding": "q6_k", "m": 1, "n": 151936, "k": 4096},
        # one token of a smaller model whose sizes are whole super-blocks and no more, one call per matrix
        _layer("decode_m1_q4_k_2560", "linear", "q4_k", "q6_k", 2560, 640, 6912, 1, 4),
        # four sequences decoded together (or four tokens verified)
        _layer("decode_m4_q4_k_4096", "group", "q4_k", "q6_k", 4096, 1024, 12288, 4, 2),
        # eight sequences on the 8-bit encoding
        _layer("decode_m8_q8_0_4096", "linear", "q8_0", "q8_0", 4096, 1024, 12288, 8, 1),
        # an odd batch on a 32-element encoding
        _layer("decode_m3_q5_0_3072", "linear", "q5_0", "q5_0", 3072, 1024, 8192, 3, 2),
        # a short prompt, or speculative tokens of several sequences
        _layer("chunk_m32_q4_k_4096", "group", "q4_k", "q6_k", 4096, 1024, 12288, 32, 2),
        # a ragged prompt on one of the small encodings, one call per matrix
        _layer("prefill_m333_q3_k_2560", "linear", "q3_k", "q3_k", 2560, 640, 6912, 333, 1),
        # an ordinary prompt
        _layer("prefill_m512_q4_k_4096", "group", "q4_k", "q6_k", 4096, 1024, 12288, 512, 1),
        # a long prompt's chunk: the most work of one pass
        _layer("prefill_m2048_q4_k_4096", "group", "q4_k", "q6_k", 4096, 1024, 12288, 2048, 1),
        # weights materialised for another library
        {"name": "dequant_q6_k_12288x4096", "op": "dequant", "encoding": "q6_k", "n": 12288, "k": 4096,
         "out": "float16", "count": 2},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _multiple(rng, low, high, step):
    return max(1, round(_log_int(rng, low, high) / step)) * step


def draw(rng):
    kind = rng.choice(("packed", "head", "decode", "decode", "decode", "chunk", "prefill", "dequant"))
    encoding = rng.choice(("q4_k", "q4_k", "q6_k", "q8_0", "q4_0", *sorted(GEOMETRY)))
    qk = GEOMETRY[encoding][0]
    if kind == "packed":
        return {"op": "packed", "encoding": encoding, "m": rng.choice((1, 1, _log_int(rng, 2, 64))),
                "n": _log_int(rng, 256, 4096), "k": _multiple(rng, 512, 4096, qk)}
    if kind == "head":
        return {"op": "head", "encoding": encoding, "m": rng.choice((1, 1, rng.randint(2, 8))),
                "n": _log_int(rng, 32000, 151936), "k": _multiple(rng, 1024, 4096, qk)}
    if kind == "dequant":
        return {"op": "dequant", "encoding": encoding, "n": _log_int(rng, 1024, 16384),
                "k": _multiple(rng, 1024, 8192, qk), "out": rng.choice(("float16", "float32")), "count": rng.randint(1, 2)}
    down = "q6_k" if encoding in ("q3_k", "q4_k", "q5_k") and rng.random() < 0.5 else encoding
    hidden = _multiple(rng, 1024, 6144, qk)
    case = {"op": "layer", "entry": rng.choice(("linear", "group")), "encoding": encoding, "down": down,
            "hidden": hidden, "kv": max(64, hidden // rng.choice((1, 4, 8))),
            "ffn": _multiple(rng, 2 * hidden, min(3.5 * hidden, 16384), qk)}
    if kind == "decode":
        case["m"] = rng.choice((1, 1, rng.randint(2, 8), rng.randint(2, 8)))
        case["layers"] = max(1, min(6, round(200e6 / sum(_bytes(e, n, k) for e, n, k in _matrices(case)))))
    else:
        weights = sum(n * k for _, n, k in _matrices(case))
        rows = int(1e11 / weights)  # small models take longer prompts, so that a pass costs less than the largest
        case["m"] = rng.randint(9, 128) if kind == "chunk" else _log_int(rng, 129, min(2048, max(160, rows)))
        case["layers"] = 1
    return case


# ------------------------------------------------------------------ sizes

def _bytes(encoding, n, k):
    qk, block = GEOMETRY[encoding]
    return n * (k // qk) * block


def _matrices(case):
    """(encoding, rows, columns) of q, k, v, o, gate, up and down."""
    h, kv, f, e = case["hidden"], case["kv"], case["ffn"], case["encoding"]
    return [(e, h, h), (e, kv, h), (e, kv, h), (e, h, h), (e, f, h), (e, f, h), (case["down"], h, f)]


def work(case):
    if case["op"] == "dequant":
        items = case["n"] * case["k"]
        size = 2 if case["out"] == "float16" else 4
        return {"bytes": case["count"] * (_bytes(case["encoding"], case["n"], case["k"]) + size * items),
                "flops": case["count"] * items}
    if case["op"] in ("packed", "head"):
        e, m, n, k = (case[key] for key in ("encoding", "m", "n", "k"))
        return {"bytes": _bytes(e, n, k) + m * k * (4 if case["op"] == "packed" else 2) + 4 * m * n,
                "flops": 2 * m * n * k}
    m, h, kv, f = case["m"], case["hidden"], case["kv"], case["ffn"]
    fused = case["entry"] == "group" and m <= GEMV_ROWS
    values = m * (3 * h + f) + m * (h + 2 * kv + h + (f if fused else 2 * f) + h)
    total = sum(_bytes(*each) for each in _matrices(case)) + 2 * values
    return {"bytes": case["layers"] * total,
            "flops": case["layers"] * sum(2 * m * n * k for _, n, k in _matrices(case))}


def tolerance(case):
    if case["op"] == "dequant":
        return "exact"  # every product is exact, and at most one sum and one cast are rounded
    # four times what the path measures against exact(), by what is rounded
    if case["m"] > GEMV_ROWS or (case["op"] == "packed" and case["m"] > 1):
        return {"rel": 1.2e-3}  # weights and activations to fp16, fp16 output: 3.0e-4
    if case["op"] in ("packed", "head"):
        return {"rel": 6e-5}  # fp32 sums and output: 1e-7 to 1.5e-5, by encoding and rows
    return {"rel": 9e-4}  # fp32 sums, fp16 output: 2.2e-4


# ----------------------------------------------------------------- inputs

def _set_half(blocks, offset, values):
    blocks[:, offset:offset + 2] = values.to(torch.float16).view(torch.uint8).view(-1, 2)


def _weight(generator, encoding, n, k):
    """Raw rows [n, row bytes]: random codes, scales for weights of zero mean and deviation 0.02
    or so, as a quantizer leaves them (minimums at the centre of the codes' range)."""
    qk, size = GEOMETRY[encoding]
    blocks = torch.randint(0, 256, (n * (k // qk), size), dtype=torch.uint8, device="cuda", generator=generator)
    spread = {"q4_0": 4.6, "q4_1": 4.6, "q5_0": 9.2, "q5_1": 9.2, "q8_0": 74.0, "q2_k": 13.0, "q3_k": 42.0,
              "q4_k": 223.0, "q5_k": 447.0, "q6_k": 1369.0}[encoding]  # deviation of (scale times) code
    d = (0.02 / spread) * (0.75 + 0.5 * torch.rand(blocks.shape[0], device="cuda", generator=generator))
    if encoding in ("q4_0", "q5_0", "q8_0"):
        _set_half(blocks, 0, d)
    elif encoding in ("q4_1", "q5_1"):
        _set_half(blocks, 0, d)
        _set_half(blocks, 2, d * (-7.5 if encoding == "q4_1" else -15.5))
    elif encoding == "q2_k":
        scales = (blocks[:, :16] & 15) | 8
        blocks[:, :16] = scales | (scales << 4)
        _set_half(blocks, 80, d)
        _set_half(blocks, 82, 1.5 * d)
    elif encoding == "q3_k":
        _set_half(blocks, 108, d)
    elif encoding == "q6_k":
        _set_half(blocks, 208, d)
    else:  # q4_k, q5_k: six-bit scales of 32 to 63, each minimum's code that of its scale
        blocks[:, 4:8] |= 0xA0
        blocks[:, 8:12] = blocks[:, 4:8]
        blocks[:, 12:16] = (blocks[:, 12:16] & 15) * 17
        _set_half(blocks, 0, d)
        _set_half(blocks, 2, d * (7.5 if encoding == "q4_k" else 15.5))
    return blocks.view(n, (k // qk) * size)


def _activation(generator, m, k, dtype):
    return torch.randn((m, k), device="cuda", generator=generator).to(dtype)


def _inputs(case, seed):
    """Weights and activations of a case from the seed alone, in the order its outputs come."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    if case["op"] == "dequant":
        return [(case["encoding"], _weight(g, case["encoding"], case["n"], case["k"]), None)
                for _ in range(case["count"])]
    if case["op"] in ("packed", "head"):
        dtype = torch.float32 if case["op"] == "packed" else torch.float16
        return [(case["encoding"], _weight(g, case["encoding"], case["n"], case["k"]),
                 _activation(g, case["m"], case["k"], dtype))]
    result = []
    for _ in range(case["layers"]):
        m, h = case["m"], case["hidden"]
        attention, output, mlp = (_activation(g, m, h, torch.float16) for _ in range(3))
        x = [attention] * 3 + [output] + [mlp] * 2 + [_activation(g, m, case["ffn"], torch.float16)]
        result += [(e, _weight(g, e, n, k), x[i]) for i, (e, n, k) in enumerate(_matrices(case))]
    return result


@functools.lru_cache(maxsize=None)
def _kernel(name, encoding, out_dtype, count=None, shape=None):
    options = {"encoding": encoding, "out_dtype": out_dtype}
    if count:
        options["count"] = count
    if shape:
        options.update(zip("mnk", shape))
    return tt.load(name, **options)


@functools.lru_cache(maxsize=None)
def _dequant(encoding, out_dtype):
    return session(0).load("gguf_dequant", encoding=encoding, out_dtype=out_dtype)


def prepare(case, seed):
    inputs = _inputs(case, seed)
    if case["op"] == "dequant":  # K is no shape of an argument: bound on the provider's own buffers
        device = session(0)
        kernel = _dequant(case["encoding"], case["out"])
        outputs = [torch.empty((case["n"], case["k"]), dtype=getattr(torch, case["out"]), device="cuda") for _ in inputs]
        calls = [kernel.bind(device.from_dlpack(w), device.from_dlpack(out)) for (_, w, _), out in zip(inputs, outputs)]
        return {"calls": [call.launch for call in calls], "outputs": outputs}
    if case["op"] == "packed":
        (encoding, w, x), = inputs
        kernel = _kernel("gguf_linear", encoding, "float32", shape=(case["m"], case["n"], case["k"]))
        calls = [kernel.prepare(x.view(-1), w.view(-1))]
    elif case["op"] == "head":
        (encoding, w, x), = inputs
        calls = [_kernel("gguf_linear", encoding, "float32").prepare(x, w)]
    elif case["entry"] == "linear":
        calls = [_kernel("gguf_linear", e, "float16").prepare(x, w) for e, w, x in inputs]
    else:
        calls = []
        scratch = {}
        for i in range(0, len(inputs), 7):
            q, k, v, o, gate, up, down = inputs[i:i + 7]
            if case["m"] <= GEMV_ROWS:
                calls.append(_kernel("gguf_gemv_group", q[0], "float16", 3).prepare(q[2], q[1], k[1], v[1]))
                calls.append(_kernel("gguf_linear", o[0], "float16").prepare(o[2], o[1]))
                calls.append(_kernel("gguf_gemv_swiglu", gate[0], "float16").prepare(gate[2], gate[1], up[1]))
                calls.append(_kernel("gguf_linear", down[0], "float16").prepare(down[2], down[1]))
            else:
                for group in ((q, k, v), (o,), (gate, up), (down,)):
                    encoding, x, weights = group[0][0], group[0][2], [w for _, w, _ in group]
                    need = session(0).gemm_workspace(encoding, case["m"], x.shape[1], [w.shape[0] for w in weights])
                    need = max(need, 256)
                    if need not in scratch:
                        scratch[need] = torch.empty(need, dtype=torch.uint8, device="cuda")
                    kernel = _kernel("gguf_gemm_group", encoding, "float16", len(weights))
                    calls.append(kernel.prepare(x, *weights, scratch[need]))
    return {"calls": calls, "outputs": [out for call in calls for out in call.outputs]}


def run(state):
    for call in state["calls"]:
        call()
    return state["outputs"]


# ------------------------------------------------------- the same in 64 bits

def _half(blocks, offset):
    return blocks[..., offset:offset + 2].contiguous().view(torch.float16).to(torch.float64)


def _six_bit(scales):
    """The eight scales and eight minimums of a 12-byte K-quant header."""
    a, b, c = scales[..., 0:4], scales[..., 4:8], scales[..., 8:12]
    return (torch.cat([a & 63, (c & 15) | ((a >> 6) << 4)], -1).double(),
            torch.cat([b & 63, (c >> 4) | ((b >> 6) << 4)], -1).double())


def _decode(encoding, raw):
    """fp64 weights [rows, columns] of raw rows, from the block layouts."""
    qk, size = GEOMETRY[encoding]
    b = raw.reshape(raw.shape[0], -1, size)
    shape = b.shape[:2]

    def nibbles(q):  # low nibbles, then high nibbles
        return torch.cat([q & 15, q >> 4], -1)

    if encoding == "q8_0":
        w = b[..., 2:].contiguous().view(torch.int8).double() * _half(b, 0)
    elif encoding == "q4_0":
        w = (nibbles(b[..., 2:]).double() - 8) * _half(b, 0)
    elif encoding == "q4_1":
        w = nibbles(b[..., 4:]).double() * _half(b, 0) + _half(b, 2)
    elif encoding in ("q5_0", "q5_1"):
        at = 2 if encoding == "q5_0" else 4
        bits = torch.arange(8, device=raw.device, dtype=torch.uint8)
        fifth = ((b[..., at:at + 4, None] >> bits) & 1).reshape(*shape, 32)
        q = (nibbles(b[..., at + 4:]) | (fifth << 4)).double()
        w = (q - 16) * _half(b, 0) if encoding == "q5_0" else q * _half(b, 0) + _half(b, 2)
    elif encoding in ("q2_k", "q3_k"):
        at = 16 if encoding == "q2_k" else 32
        two = torch.tensor([0, 2, 4, 6], device=raw.device, dtype=torch.uint8)[:, None]
        codes = (b[..., at:at + 64].reshape(*shape, 2, 1, 32) >> two) & 3  # [half, plane, 32]
        if encoding == "q2_k":
            scale, low = (b[..., :16] & 15).double() * _half(b, 80), (b[..., :16] >> 4).double() * _half(b, 82)
            w = codes.reshape(*shape, 16, 16).double() * scale[..., None] - low[..., None]
        else:
            bits = torch.arange(8, device=raw.device, dtype=torch.uint8).reshape(2, 4, 1)
            high = (b[..., :32].reshape(*shape, 1, 1, 32) >> bits) & 1
            packed, top = b[..., 96:104], b[..., 104:108]
            low = torch.cat([packed & 15, packed >> 4], -1)
            high2 = torch.cat([(top >> s) & 3 for s in (0, 2, 4, 6)], -1)
            scale = ((low | (high2 << 4)).double() - 32) * _half(b, 108)
            w = (codes.double() - 4 * (1 - high.double())).reshape(*shape, 16, 16) * scale[..., None]
    elif encoding in ("q4_k", "q5_k"):
        scale, low = _six_bit(b[..., 4:16])
        scale, low = scale * _half(b, 0), low * _half(b, 2)
        q = b[..., -128:].reshape(*shape, 4, 32)
        codes = torch.stack([q & 15, q >> 4], -2).reshape(*shape, 8, 32)
        if encoding == "q5_k":
            bits = torch.arange(8, device=raw.device, dtype=torch.uint8)[:, None]
            codes = codes | (((b[..., None, 16:48] >> bits) & 1) << 4)
        w = codes.double() * scale[..., None] - low[..., None]
    else:  # q6_k
        ql = b[..., :128].reshape(*shape, 2, 1, 64)
        lows = torch.cat([ql & 15, ql >> 4], -2).reshape(*shape, 2, 4, 32)
        two = torch.tensor([0, 2, 4, 6], device=raw.device, dtype=torch.uint8)[:, None]
        highs = (b[..., 128:192].reshape(*shape, 2, 1, 32) >> two) & 3
        scale = b[..., 192:208].contiguous().view(torch.int8).double() * _half(b, 208)
        w = ((lows | (highs << 4)).double() - 32).reshape(*shape, 16, 16) * scale[..., None]
    return w.reshape(raw.shape[0], -1)


def _product(encoding, w, x):
    x = x.double()
    return torch.cat([x @ _decode(encoding, rows).T for rows in w.split(8192)], 1)


def exact(case, seed):
    inputs = _inputs(case, seed)
    if case["op"] == "dequant":
        return [_decode(e, w) for e, w, _ in inputs]
    products = [_product(*each) for each in inputs]
    if case["op"] == "packed":
        return [products[0].view(-1)]
    if case["op"] == "layer" and case["entry"] == "group" and case["m"] <= GEMV_ROWS:
        result = []
        for i in range(0, len(products), 7):
            q, k, v, o, gate, up, down = products[i:i + 7]
            result += [q, k, v, o, gate * torch.sigmoid(gate) * up, down]
        return result
    return products
