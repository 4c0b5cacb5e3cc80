"""Timing cases of the framework: what a program that serves quantized models has it do, through its public entry points.

Every case is a compiled graph that is launched on its resident buffers (Session.compile, set_param_typed, launch), or one that
is run on host arrays (CompiledGraph.run), or the LM-head call of the C ABI. Weights are GGUF blocks of ~N(0, 0.02) values,
activations are ~N(0, 1). All states share one stream, as the layers of a model do.

kinds
  matmul  x [m, k] times the matrices of `n` (several: projections that share their input), packed in `scheme`; `host`: through
          run() with arrays in and out, else resident
  layer   the matmul path of a decoder layer in data-flow order: norm -> q, k, v; q -> o; norm -> up | gate -> SwiGLU -> down
          (attention itself is not an operator of this framework: o reads q); f32 activations
  fq      FakeQuantize of [rows, k], per channel along `axis`
  chain   FakeQuantize of [m, k] per column, then a matmul by an [n, k] matrix
  topk    the `cap` best logits of a tied LM head [n, k] for one hidden vector
  moe     m routed rows times the [n, k] matrices of `experts` experts
"""
import ctypes
import math

import numpy as np
import torch

import rlx_amd
from rlx_amd import DType, Graph, Op, QuantScheme, Session, Shape, ops

SCHEMES = {"q4_0": QuantScheme.GgufQ4_0, "q8_0": QuantScheme.GgufQ8_0, "q4_k": QuantScheme.GgufQ4K, "q5_k": QuantScheme.GgufQ5K,
           "q6_k": QuantScheme.GgufQ6K, "q8_k": QuantScheme.GgufQ8K, "q2_k": QuantScheme.GgufQ2K, "q3_k": QuantScheme.GgufQ3K}
DTYPES = {"f32": (DType.F32, torch.float32), "bf16": (DType.BF16, torch.bfloat16), "f16": (DType.F16, torch.float16)}
EPS = 1e-5


def listed():
    return [
        # the smallest call: one attention-sized projection of one token
        {"name": "gemv", "kind": "matmul", "scheme": "q8_0", "dtype": "f32", "m": 1, "k": 4096, "n": "4096", "host": False},
        # three projections of a smaller model through the host boundary, sizes that fill no tile evenly, a scheme with wide super-blocks
        {"name": "host_call", "kind": "matmul", "scheme": "q6_k", "dtype": "f32", "m": 3, "k": 2304, "n": "2310,770,770", "host": True},
        # one token through a Llama-3-8B layer: what a decode loop repeats per layer
        {"name": "decode_layer", "kind": "layer", "scheme": "q4_0", "m": 1, "k": 4096, "kv": 1024, "ffn": 14336},
        # the same layer for six sequences decoded together
        {"name": "decode_layer_batch", "kind": "layer", "scheme": "q4_k", "m": 6, "k": 4096, "kv": 1024, "ffn": 14336},
        # Llama-3-70B projections for a decode batch of 16, and for 64 rows, where decoding turns into prefill
        {"name": "batch_16", "kind": "matmul", "scheme": "q4_0", "dtype": "bf16", "m": 16, "k": 8192, "n": "28672", "host": False},
        {"name": "batch_64", "kind": "matmul", "scheme": "q4_0", "dtype": "bf16", "m": 64, "k": 28672, "n": "8192", "host": False},
        # gate and up of a Llama-3-8B layer for a prompt of 512 tokens
        {"name": "prefill", "kind": "matmul", "scheme": "q4_k", "dtype": "bf16", "m": 512, "k": 4096, "n": "14336,14336", "host": False},
        # a longer prompt, of no round length, through the whole layer: activations stay f32 from one operator to the next
        {"name": "prefill_layer", "kind": "layer", "scheme": "q4_0", "m": 1111, "k": 4096, "kv": 1024, "ffn": 14336},
        # quantization-aware evaluation: activations of 8192 tokens to int8 per channel, alone and into a matmul
        {"name": "fake_quant", "kind": "fq", "m": 8192, "k": 4096, "axis": 1, "bits": 8},
        {"name": "fake_quant_matmul", "kind": "chain", "scheme": "q8_0", "m": 8192, "k": 4096, "n": "4096"},
        # the last step of a token: the best 40 of a Llama-3 vocabulary for the sampler
        {"name": "lm_head", "kind": "topk", "scheme": "q4_k", "k": 4096, "n": "128256", "cap": 40},
        # 512 tokens routed to two of eight experts each
        {"name": "experts", "kind": "moe", "scheme": "q4_0", "dtype": "f16", "m": 1024, "k": 4096, "n": "14336", "experts": 8},
    ]


MOST_WEIGHTS = 8 * 14336 * 4096   # of the largest listed cases
MOST_FLOPS = 4.5e11
MOST_F32_FLOPS = 2.2e11           # an f32 activation counts twice on the matrix cores


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cols(rng, scheme, lo, hi):
    """A row length of whole blocks, odd numbers of blocks among them."""
    block = SCHEMES[scheme].gguf_block_size()
    return max(1, _log(rng, lo, hi) // block) * block


def draw(rng):
    while True:
        kind = rng.choice(["matmul", "matmul", "matmul", "matmul", "layer", "layer", "fq", "chain", "topk", "moe"])
        scheme = rng.choice(["q4_0", "q4_0", "q8_0", "q8_0", "q4_k", "q4_k", "q6_k", "q5_k", "q8_k", "q2_k", "q3_k"])
        dtype = rng.choice(list(DTYPES))
        if kind == "matmul":
            host = rng.random() < 0.2
            m = _log(rng, 1, 8) if host else _log(rng, 1, 32) if rng.random() < 0.5 else _log(rng, 33, 4096)
            count = rng.choice([1, 1, 2, 3])
            c = {"kind": kind, "scheme": scheme, "dtype": "f32" if host else dtype, "m": m, "k": _cols(rng, scheme, 768, 28672),
                 "n": ",".join(str(_log(rng, 512, 28672)) for _ in range(count)), "host": host}
        elif kind == "layer":
            k = _log(rng, 4, 16) * 256
            c = {"kind": kind, "scheme": scheme, "m": _log(rng, 1, 8) if rng.random() < 0.5 else _log(rng, 9, 1024), "k": k,
                 "kv": k // rng.choice([1, 2, 4, 8]), "ffn": _log(rng, 2 * k // 256, min(56, 4 * k // 256)) * 256}
        elif kind == "fq":
            c = {"kind": kind, "m": _log(rng, 64, 8192), "k": _log(rng, 64, 4096), "axis": rng.choice([0, 1, 1]), "bits": rng.choice([8, 8, 4])}
        elif kind == "chain":
            c = {"kind": kind, "scheme": rng.choice(["q8_0", "q4_0"]), "m": _log(rng, 64, 8192), "k": _cols(rng, "q8_0", 512, 4096), "n": str(_log(rng, 512, 4096))}
        elif kind == "topk":
            c = {"kind": kind, "scheme": rng.choice(["q4_k", "q6_k", "q8_0"]), "k": 256 * _log(rng, 4, 16), "n": str(_log(rng, 8000, 128256)), "cap": _log(rng, 1, 64)}
        else:
            experts = rng.choice([4, 8, 16, 32])
            c = {"kind": kind, "scheme": rng.choice(["q4_0", "q8_0", "q4_k"]), "dtype": dtype, "m": _log(rng, 2, 2048), "k": 256 * _log(rng, 2, 16),
                 "n": str(_log(rng, 512, 14336)), "experts": experts}
        flops = work(c)["flops"]
        slow = 3 if c.get("scheme") in ("q5_k", "q6_k", "q3_k", "q2_k") else 1  # schemes whose upload takes longer
        if _weights(c) * slow <= MOST_WEIGHTS and flops <= (MOST_FLOPS if c.get("dtype", "f32") != "f32" or kind == "chain" or c["kind"] == "fq" else MOST_F32_FLOPS):
            return c


def _ns(case):
    return [int(v) for v in case["n"].split(",")]


def _matrices(case):
    """(rows, columns) of the packed matrices of a case."""
    if case["kind"] == "fq":
        return []
    if case["kind"] == "layer":
        k, kv, ffn = case["k"], case["kv"], case["ffn"]
        return [(k, k), (kv, k), (kv, k), (k, k), (2 * ffn, k), (k, ffn)]
    return [(n, case["k"]) for n in _ns(case)] * case.get("experts", 1)


def _weights(case):
    return sum(n * k for n, k in _matrices(case))


def work(case):
    m, k = case.get("m", 1), case["k"]
    if case["kind"] == "fq":
        return {"bytes": 8 * m * k, "flops": 4 * m * k}
    scheme = SCHEMES[case["scheme"]]
    packed = _weights(case) // scheme.gguf_block_size() * scheme.gguf_block_bytes()
    x_bytes = m * k * (2 if case.get("dtype", "f32") != "f32" else 4)
    if case["kind"] == "layer":
        out = 4 * m * (2 * k + 2 * case["kv"])
    elif case["kind"] == "topk":
        out = 8 * case["cap"]
    else:
        out = 4 * m * sum(_ns(case))
    if case["kind"] == "moe":  # a row meets one expert, and few rows do not meet them all
        packed = packed * min(m, case["experts"]) // case["experts"]
    flops = 2.0 * m * (_ns(case)[0] * k if case["kind"] == "moe" else _weights(case))
    return {"bytes": packed + x_bytes + out, "flops": flops}


def tolerance(case):
    """Four times what the outputs measured against 64-bit products of the decoded weights. Where every weight code and block scale
    is multiplied exactly, f32 sums remain; Q6_K at every size, and Q4_0 / Q8_0 above the decode sizes, round the product of scale and
    code to the 11 bits of binary16 once."""
    kind, scheme = case["kind"], case.get("scheme")
    if kind == "fq":
        return "exact"
    decode_rows = 16 if case.get("dtype", "f32") == "f32" else 32
    rounded = scheme == "q6_k" or kind == "chain" or (scheme in ("q4_0", "q8_0") and case.get("m", 1) > decode_rows)
    if kind == "chain":
        return {"rel": 8e-4, "max": 4e-2}
    if kind == "layer":
        return {"rel": 2e-3, "max": 1e-2} if rounded else {"rel": 2.5e-6, "max": 1e-5}
    limit = {"rel": 7e-4, "max": 4e-3} if rounded else {"rel": 1e-6, "max": 6e-6}
    if kind == "topk":
        limit["differ"] = 0.01  # neighbours of almost equal value may trade places
    return limit


# ---- states ----------------------------------------------------------------------------------------------

_stream = None


def _the_stream():
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def _pool(name, rng):
    """Packed blocks of ~N(0, 0.02) weights (about a million of them): through the encoder where there is one, else block fields
    drawn so that the decoded values have that spread."""
    scheme = SCHEMES[name]
    if name in ("q4_0", "q8_0", "q4_k"):
        return ops.quantize(scheme, rng.standard_normal(1 << 20, dtype=np.float32) * np.float32(0.02)).reshape(-1, scheme.gguf_block_bytes())
    blocks = (1 << 20) // 256
    p = rng.integers(0, 256, (blocks, scheme.gguf_block_bytes()), dtype=np.uint8)

    def put(at, values, kind):
        raw = values.astype(kind).view(np.uint8).reshape(blocks, -1)
        p[:, at:at + raw.shape[1]] = raw

    spread = rng.uniform(0.6, 1.4, blocks)
    if name == "q6_k":    # d * sc * (q - 32)
        p[:, 192:208] = rng.integers(32, 128, (blocks, 16), dtype=np.uint8)
        put(208, 0.02 / (84 * 18.5) * spread, np.float16)
    elif name == "q8_k":  # d * q
        put(0, 0.02 / 74 * spread, np.float32)
    elif name == "q3_k":  # d * (sc - 32) * code
        put(0, 0.02 / (18.5 * 2.3) * spread, np.float16)
    elif name == "q5_k":  # sc * (d * q - dmin), the minimum in the middle of the codes
        d = 0.02 / (36 * 9.2) * spread
        put(0, d, np.float16)
        put(2, 15.5 * d, np.float16)
        p[:, 8:12] = p[:, 4:8]
        p[:, 12:16] = (p[:, 12:16] & 0xF) * 17
    else:                 # q2_k: sc * (d * q - dmin)
        d = 0.02 / (8.8 * 1.12) * spread
        put(0, d, np.float16)
        put(2, 1.5 * d, np.float16)
        p[:, 4:20] = (p[:, 4:20] & 0xF) * 17
    return p


def _packed(pool, name, n, k, rng):
    """[n, k] packed rows: blocks of the pool in random order."""
    count = n * k // SCHEMES[name].gguf_block_size()
    return pool[rng.integers(0, len(pool), count, dtype=np.int32)].reshape(-1)


class _DeviceBytes:
    def __init__(self, ptr, nbytes):
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (ptr, False), "version": 2}


def _view(graph, ptr, shape, dtype):
    nbytes = math.prod(shape) * torch.empty(0, dtype=dtype).element_size()
    tensor = torch.as_tensor(_DeviceBytes(ptr, nbytes), device="cuda").view(dtype).view(*shape)
    tensor.graph = graph  # whose buffer this is: it lives as long as the tensor does
    return tensor


def _slot(graph, name, shape, dtype):
    """A tensor over the buffer of an input or parameter."""
    p, n = ctypes.c_void_p(), ctypes.c_size_t()
    rlx_amd._lib.check(rlx_amd._lib.lib().rlx_exec_slot(graph._h, name.encode(), ctypes.byref(p), ctypes.byref(n)))
    return _view(graph, p.value, shape, dtype)


def _output(graph, i, shape):
    p, n = ctypes.c_void_p(), ctypes.c_size_t()
    rlx_amd._lib.check(rlx_amd._lib.lib().rlx_exec_output_slot(graph._h, i, ctypes.byref(p), ctypes.byref(n)))
    return _view(graph, p.value, shape, torch.float32)


def _normal(seed, shape, dtype=torch.float32):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


def _build(case):
    """(graph, [(weight name, rows, columns)], output shapes)"""
    g = Graph.new(case["kind"])
    m, k, kind = case["m"], case["k"], case["kind"]
    weights = []
    scheme = SCHEMES.get(case.get("scheme"))

    def packed(name, n, kk, stack=1):
        weights.append((name, n * stack, kk))
        return g.param(name, Shape.new([stack * n * kk // scheme.gguf_block_size() * scheme.gguf_block_bytes()], DType.U8))

    def matmul(x, name, n, kk):
        return g.add_node(Op.DequantMatMul(scheme), [x, packed(name, n, kk)], Shape.new([m, n], DType.F32))

    dt = DTYPES[case.get("dtype", "f32")][0]
    x = g.input("x", Shape.new([m, k], dt))
    if kind == "matmul":
        outs = [matmul(x, "w%d" % i, n, k) for i, n in enumerate(_ns(case))]
    elif kind == "layer":
        kv, ffn = case["kv"], case["ffn"]
        gammas = [g.param(name, Shape.new([k], DType.F32)) for name in ("gamma0", "gamma1")]
        h = g.add_node(Op.RmsNorm(EPS), [x, gammas[0]], Shape.new([m, k], DType.F32))
        q, key, val = matmul(h, "wq", k, k), matmul(h, "wk", kv, k), matmul(h, "wv", kv, k)
        o = matmul(q, "wo", k, k)
        h = g.add_node(Op.RmsNorm(EPS), [o, gammas[1]], Shape.new([m, k], DType.F32))
        act = g.fused_swiglu(matmul(h, "wup_gate", 2 * ffn, k))
        outs = [o, key, val, matmul(act, "wdown", k, ffn)]
    elif kind == "moe":
        idx = g.input("expert", Shape.new([m], DType.F32))
        n = _ns(case)[0]
        outs = [g.dequant_grouped_matmul(x, packed("w", n, k, case["experts"]), idx, scheme, Shape.new([m, n], DType.F32))]
    else:
        q = g.fake_quantize(x, case.get("bits", 8), case.get("axis", 1))
        outs = [q] if kind == "fq" else [matmul(q, "w", _ns(case)[0], k)]
    g.set_outputs(outs)
    return g, weights, [g.nodes[o].shape.dims for o in outs]


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    pool = _pool(case["scheme"], rng) if "scheme" in case else None
    stream = _the_stream()
    if case["kind"] == "topk":
        n, k, cap = _ns(case)[0], case["k"], case["cap"]
        weight = ops.QWeight(SCHEMES[case["scheme"]], _packed(pool, case["scheme"], n, k, rng), n, k)
        need = rlx_amd._lib.lib().rlx_mi355x_tied_lm_topk_scratch_bytes(n, cap)
        state = {"call": "topk", "weight": weight, "hidden": _normal(seed, (k,)), "cap": cap, "stream": stream.cuda_stream, "need": need,
                 "scratch": torch.empty(need, dtype=torch.uint8, device="cuda"),
                 "rows": torch.empty(cap, dtype=torch.int32, device="cuda"), "values": torch.empty(cap, dtype=torch.float32, device="cuda")}
        torch.cuda.synchronize()
        return state
    graph, weights, shapes = _build(case)
    c = Session.new(rlx_amd.Device.Mi355x).compile(graph)
    c.set_stream(stream.cuda_stream)
    for name, n, k in weights:
        c.set_param_typed(name, _packed(pool, case["scheme"], n, k, rng), DType.U8)
    m, k = case["m"], case["k"]
    if case["kind"] == "layer":
        for name in ("gamma0", "gamma1"):
            c.set_param(name, (1 + 0.1 * rng.standard_normal(k)).astype(np.float32))
    if case.get("host"):
        return {"call": "run", "graph": c, "shapes": shapes, "inputs": [("x", rng.standard_normal((m, k), dtype=np.float32))]}
    x = _normal(seed, (m, k), DTYPES[case.get("dtype", "f32")][1])
    if case["kind"] in ("fq", "chain"):  # heavy tails: one value in a thousand twenty times larger
        tail = torch.rand((m, k), generator=torch.Generator(device="cuda").manual_seed(seed + 1), device="cuda") < 0.001
        x = torch.where(tail, x * 20, x)
    _slot(c, "x", (m, k), x.dtype).copy_(x)
    if case["kind"] == "moe":  # every expert takes part; some get more rows than others
        share = rng.dirichlet(np.full(case["experts"], 8.0))
        route = torch.from_numpy(rng.choice(case["experts"], m, p=share).astype(np.float32))
        _slot(c, "expert", (m,), torch.float32).copy_(route)
    torch.cuda.synchronize()
    return {"call": "launch", "graph": c, "outputs": [_output(c, i, shape) for i, shape in enumerate(shapes)]}


def run(state):
    if state["call"] == "launch":
        state["graph"].launch()
        return state["outputs"]
    if state["call"] == "run":
        return state["graph"].run(state["inputs"])
    rlx_amd._lib.check(rlx_amd._lib.lib().rlx_mi355x_gguf_tied_lm_topk(
        state["hidden"].data_ptr(), int(DType.F32), state["weight"].ptr, state["cap"], state["rows"].data_ptr(), state["values"].data_ptr(),
        state["scratch"].data_ptr(), state["need"], state["stream"]))
    return state["rows"], state["values"]
