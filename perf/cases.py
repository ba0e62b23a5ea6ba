"""What a user of the library has it do, as timed cases: the quantized matmuls of whole decode steps and
prefills, an encoder through the backend object, and the row operators of loading and cache writes.

A case is a dict of plain values:

  kind "linear"   one call of the plain op, as a host calls it between its own kernels
  kind "decoder"  every matmul of `layers` decoder layers on `rows` tokens: the attention input projection (one fused
                  matrix of `qkv` columns; with `kv` > 0 a query matrix of `qkv` columns and a key / value pair of `kv`
                  columns each), the attention output projection, gate and up as one pair call, down; with `vocab` > 0
                  the greedy head on the last row.  `graph`: the step is captured once and replayed, as a decode loop does
  kind "encoder"  `layers` encoder layers with biases through the backend object: Q/K/V as one triple, output projection
                  plus residual, first FFN matrix with gelu, second plus residual
  kind "rows"     the row operators on a [rows, dim] table: quantize all of it, dequantize all of it, look up `lookups`
                  rows

Weights are normal values quantized by the library's own quantizers, so block scales and quants are distributed as in a
quantized checkpoint.  Activations are normal with a few large channels (what enters the attention and gate / up matmuls)
or products of two normals (what enters the down matmul); every matmul has inputs of its own, as the norms, rotations and
softmaxes that lie between them are not this library's.
"""
from __future__ import annotations

import torch

from antfly_amd import _lib, kernels
from antfly_amd._lib import Buffer
from antfly_amd.hip_compute import HipCompute

FORMATS = {"q4_0": _lib.TYPE_Q4_0, "q8_0": _lib.TYPE_Q8_0, "q4_k": _lib.TYPE_Q4_K}
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144)}
DEVICE = "cuda:0"


def _decoder(name, fmt, rows, layers, hidden, qkv, ffn, kv=0, vocab=0, graph=False):
    case = {"kind": "decoder", "fmt": fmt, "rows": rows, "layers": layers, "hidden": hidden, "qkv": qkv, "kv": kv,
            "ffn": ffn, "vocab": vocab, "graph": graph}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one attention output projection of a decode step, called by itself: the smallest call, host and launch time count
        {"name": "call_q4_0_m1", "kind": "linear", "fmt": "q4_0", "rows": 1, "in_dim": 4096, "out_dim": 4096},
        # one token of an 8B-sized decoder, greedy head included: the decode loop of a chat
        _decoder("decode_q4_0_m1", "q4_0", 1, 32, 4096, 6144, 14336, vocab=128256, graph=True),
        # the verification step of speculative decoding: four drafts and one more token
        _decoder("verify_q4_0_m5", "q4_0", 5, 32, 4096, 6144, 14336, graph=True),
        # one token of a small decoder with narrow key / value heads: many short launches
        _decoder("decode_small_q8_0_m1", "q8_0", 1, 22, 2048, 2048, 5632, kv=256, vocab=32000, graph=True),
        # one token in the K-quant format
        _decoder("decode_q4_k_m1", "q4_k", 1, 16, 4096, 6144, 14336, graph=True),
        # batched decode: 32 requests, one token each
        _decoder("batch_q4_0_m32", "q4_0", 32, 8, 4096, 6144, 14336, graph=True),
        # prompt processing: a chunk of 512 tokens, 8-bit weights
        _decoder("prefill_q8_0_m512", "q8_0", 512, 2, 4096, 6144, 14336),
        # the largest chunk, 4-bit weights
        _decoder("prefill_q4_0_m2048", "q4_0", 2048, 1, 4096, 6144, 14336),
        # a prompt of ordinary, odd length in the K-quant format
        _decoder("prefill_q4_k_m333", "q4_k", 333, 1, 4096, 6144, 14336),
        # a short odd prompt on the small decoder (narrow key / value matrices take the f32 route)
        _decoder("prefill_small_q4_0_m77", "q4_0", 77, 4, 2048, 2048, 5632, kv=256),
        # a text encoder of CLIP size on its full context, biases and activations fused, through the backend object
        {"name": "encoder_q4_k_m77", "kind": "encoder", "fmt": "q4_k", "rows": 77, "layers": 4, "hidden": 768, "ffn": 3072},
        # quantizing and dequantizing a table, and the embedding lookup of a prompt
        {"name": "rows_q8_0", "kind": "rows", "fmt": "q8_0", "rows": 14336, "dim": 4096, "lookups": 512},
    ]


def _matmuls(case):
    """(count, rows, in_dim, out_dim) of every matmul of one pass."""
    m = case["rows"]
    if case["kind"] == "linear":
        return [(1, m, case["in_dim"], case["out_dim"])]
    n, h, f = case["layers"], case["hidden"], case["ffn"]
    if case["kind"] == "encoder":
        return [(4 * n, m, h, h), (n, m, h, f), (n, m, f, h)]
    shapes = [(n, m, h, case["qkv"]), (n, m, h, h), (2 * n, m, h, f), (n, m, f, h)]
    if case["kv"]:
        shapes.append((2 * n, m, h, case["kv"]))
    if case["vocab"]:
        shapes.append((1, 1, h, case["vocab"]))
    return shapes


def work(case):
    values, size = BLOCK[case["fmt"]]
    if case["kind"] == "rows":
        quantized = case["rows"] * case["dim"] // values * size
        moved = 2 * (quantized + 4 * case["rows"] * case["dim"])
        moved += case["lookups"] * case["dim"] // values * size + 4 * case["lookups"] * case["dim"]
        return {"bytes": moved, "flops": 0}
    # matmuls that share an input read it once: fused or paired projections and triples
    moved = flops = 0
    for count, m, k, n in _matmuls(case):
        moved += count * (n * (k // values) * size + 4 * m * n)
        flops += count * 2 * m * k * n
    m = case["rows"]
    if case["kind"] == "linear":
        inputs = case["in_dim"]
    elif case["kind"] == "encoder":
        inputs = case["layers"] * (5 * case["hidden"] + case["ffn"])  # of four matmuls, and two residuals
    else:
        inputs = case["layers"] * (3 * case["hidden"] + case["ffn"])
    return {"bytes": moved + 4 * (m * inputs + (case["hidden"] if case.get("vocab") else 0)), "flops": flops}


def _spread(rng, low, high):
    """A whole number from low to high, even over the logarithm."""
    return min(high, max(low, round(low * (high / low) ** rng.random())))


def draw(rng):
    kind = rng.choice(["linear", "decoder", "decoder", "decoder", "decoder", "encoder", "rows"])
    fmt = rng.choice(["q4_0", "q4_0", "q8_0", "q8_0", "q4_k"])
    block = BLOCK[fmt][0]

    def dim(low, high):
        return _spread(rng, low // block, high // block) * block

    if kind == "rows":
        return {"kind": kind, "fmt": fmt, "rows": _spread(rng, 256, 14336), "dim": dim(512, 4096),
                "lookups": _spread(rng, 16, 512)}
    if kind == "linear":
        return {"kind": kind, "fmt": fmt, "rows": _spread(rng, 1, 2048), "in_dim": dim(1024, 8192),
                "out_dim": _spread(rng, 1024, 8192)}
    if kind == "encoder":
        hidden = rng.choice([512, 768, 1024])
        return {"kind": kind, "fmt": fmt, "rows": _spread(rng, 9, 514), "layers": rng.randint(2, 6), "hidden": hidden,
                "ffn": 4 * hidden}
    # prompts, batches and single tokens alike; layers as many as one listed step's bytes and operations allow
    rows = rng.choice([1, 1, _spread(rng, 2, 8), _spread(rng, 9, 64), _spread(rng, 65, 2048), _spread(rng, 65, 2048)])
    hidden = dim(1536, 5120)
    kv = rng.choice([0, 0, 256, 512])
    ffn = dim(2 * hidden, 7 * hidden // 2)
    case = _decoder(None, fmt, rows, 1, hidden, hidden if kv else 3 * hidden // 2, ffn, kv=kv, graph=rows <= 64)
    one = work(case)
    most = min(3.0e9 / one["bytes"], 6.0e11 / one["flops"])
    case["layers"] = max(1, min(16, int(most)))
    return case


def tolerance(case):
    if case["kind"] == "rows":
        return "exact"  # bytes of the format, and one rounding per dequantized value
    # four times what the library differs from the same product in 64 bits, and from itself in another summation order
    # (up to 2048 rows, K to 14336): 1.7e-7 / 1.5e-6 with quantized activations, 5e-7 / 3.6e-6 with f32 ones
    if case["fmt"] == "q4_k":
        return {"rel": 2e-6, "max": 1.5e-5}
    return {"rel": 7e-7, "max": 6e-6}


def _buf(t):
    return Buffer(t.data_ptr(), t.numel() * t.element_size())


class _Source:
    """Seeded inputs, made on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.gen, device=DEVICE, dtype=torch.float32)

    def hidden(self, rows, dim):
        """Normalised activations: normal, about one channel in 200 twenty times larger."""
        large = torch.rand(dim, generator=self.gen, device=DEVICE) < 0.005
        return self.normal(rows, dim) * torch.where(large, 20.0, 1.0)

    def gated(self, rows, dim):
        """Gate times up: a product of two normals."""
        return self.normal(rows, dim) * self.normal(rows, dim)

    def raw_weight(self, fmt, out_dim, in_dim):
        """GGUF blocks of normal weights."""
        values, size = BLOCK[fmt]
        raw = torch.empty(out_dim * (in_dim // values) * size, dtype=torch.uint8, device=DEVICE)
        dense = self.normal(out_dim, in_dim).mul_(0.02)
        kernels.launchQuantizeRows(torch.cuda.current_stream().cuda_stream, FORMATS[fmt], _buf(raw), _buf(dense), out_dim,
                                   in_dim)
        return raw

    def weight(self, fmt, out_dim, in_dim):
        """A weight in the library's device layout."""
        raw = self.raw_weight(fmt, out_dim, in_dim)
        out = torch.empty(kernels.preparedWeightBytes(FORMATS[fmt], out_dim, in_dim), dtype=torch.uint8, device=DEVICE)
        kernels.launchPrepareWeight(torch.cuda.current_stream().cuda_stream, FORMATS[fmt], _buf(out), _buf(raw), out_dim,
                                    in_dim)
        return out


def _launch_plan(case, src):
    """The calls of one pass as (launcher, arguments behind the stream), their outputs, and what they keep alive."""
    fmt, m = FORMATS[case["fmt"]], case["rows"]
    keep, calls, shapes = [], [], []

    def held(t):
        keep.append(t)
        return _buf(t)

    def result(*shape):
        return torch.empty(*shape, dtype=torch.float32, device=DEVICE)

    if case["kind"] == "linear":
        shapes.append((m, case["in_dim"], case["out_dim"]))
    else:
        h, f = case["hidden"], case["ffn"]
        shapes += [(m, h, case["qkv"]), (m, h, h), (m, h, f), (m, f, h)]
        if case["kv"]:
            shapes.append((m, h, case["kv"]))
    scratch = max(16, max(kernels.workspaceBytes(fmt, *s) for s in shapes))
    if case.get("vocab"):
        scratch = max(scratch, kernels.linearArgmaxWorkspaceBytes(fmt, case["hidden"], case["vocab"]))
    workspace = held(torch.empty(scratch, dtype=torch.uint8, device=DEVICE))
    prepared = _lib.LAYOUT_PREPARED

    def linear(y, x, k, n):
        calls.append((kernels.launchLinearF32, (fmt, prepared, _buf(y), held(x), held(src.weight(case["fmt"], n, k)), m, k, n,
                                                workspace)))

    def pair(ya, yb, x, k, n):
        calls.append((kernels.launchLinearPairF32, (fmt, prepared, _buf(ya), _buf(yb), held(x),
                                                    held(src.weight(case["fmt"], n, k)), held(src.weight(case["fmt"], n, k)),
                                                    m, k, n, workspace)))

    if case["kind"] == "linear":
        y = result(m, case["out_dim"])
        linear(y, src.hidden(m, case["in_dim"]), case["in_dim"], case["out_dim"])
        return calls, {"y": y}, keep

    layers, kv, vocab = case["layers"], case["kv"], case["vocab"]
    out = {"qkv": result(layers, m, case["qkv"]), "attn": result(layers, m, h), "gate": result(layers, m, f),
           "up": result(layers, m, f), "down": result(layers, m, h)}
    if kv:
        out["key"], out["value"] = result(layers, m, kv), result(layers, m, kv)
    for i in range(layers):
        x = src.hidden(m, h)
        linear(out["qkv"][i], x, h, case["qkv"])
        if kv:
            pair(out["key"][i], out["value"][i], x, h, kv)
        linear(out["attn"][i], src.normal(m, h), h, h)
        pair(out["gate"][i], out["up"][i], src.hidden(m, h), h, f)
        linear(out["down"][i], src.gated(m, f), f, h)
    if vocab:
        out["token"] = torch.zeros(1, dtype=torch.int32, device=DEVICE)
        calls.append((kernels.launchLinearArgmaxLastRowF32, (fmt, prepared, _buf(out["token"]), kernels.NO_BUFFER,
                                                             held(src.hidden(m, h)), held(src.weight(case["fmt"], vocab, h)),
                                                             m, h, vocab, workspace)))
    return calls, out, keep


def _issue(calls):
    stream = torch.cuda.current_stream().cuda_stream
    for launch, arguments in calls:
        launch(stream, *arguments)


class _DeviceView:
    """A backend tensor's device memory as an array that torch can view."""

    def __init__(self, tensor, shape):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (tensor.device_ptr, False),
                                         "strides": None, "version": 3}


class _Encoder:
    """An encoder's layers on the backend object, with resident weights and biases."""

    def __init__(self, case, src):
        self.rows, self.layers, self.hidden, self.ffn = case["rows"], case["layers"], case["hidden"], case["ffn"]
        self.backend = HipCompute()
        self.inputs, self.results, self.weights = [], [], {}
        h, f = self.hidden, self.ffn
        for i in range(self.layers):
            for name, n, k in (("q", h, h), ("k", h, h), ("v", h, h), ("o", h, h), ("fc1", f, h), ("fc2", h, f)):
                raw = src.raw_weight(case["fmt"], n, k).cpu().numpy()
                self.backend.insertWeightFromLoaded(f"{i}.{name}.weight", FORMATS[case["fmt"]], raw, [n, k])
                bias = (src.normal(n) * 0.1).cpu().numpy()
                self.backend.insertWeightFromTensor(f"{i}.{name}.bias", bias, [n])
                for kind in ("weight", "bias"):
                    self.weights[f"{i}.{name}.{kind}"] = self.backend.getWeight(f"{i}.{name}.{kind}")
            # what enters the layer (normalised), the attention's result, the residual stream, the FFN (normalised), its second half
            made = (src.hidden(self.rows, h), src.normal(self.rows, h), src.normal(self.rows, h), src.hidden(self.rows, h),
                    torch.nn.functional.gelu(src.normal(self.rows, f)))
            self.inputs.append([(x, self.backend.wrapDeviceFloat32(x.data_ptr(), list(x.shape))) for x in made])

    def step(self):
        cb, m, h, f, w = self.backend, self.rows, self.hidden, self.ffn, self.weights
        for tensor in self.results:
            cb.freeTensor(tensor)  # the previous step's
        self.results, views = [], {}
        for i in range(self.layers):
            x, context, residual, mid, wide = (tensor for _, tensor in self.inputs[i])

            def weight(name, i=i):
                return w[f"{i}.{name}.weight"], w[f"{i}.{name}.bias"]

            q, k, v = cb.linearTriple(x, *weight("q"), *weight("k"), *weight("v"), m, h, h)
            attn = cb.linearAdd(context, *weight("o"), residual, m, h, h)
            up = cb.linearGelu(mid, *weight("fc1"), m, h, f)
            down = cb.linearAdd(wide, *weight("fc2"), attn, m, f, h)
            named = {"q": q, "k": k, "v": v, "attn": attn, "up": up, "down": down}
            self.results += named.values()
            for name, tensor in named.items():
                views[f"{i}.{name}"] = torch.as_tensor(_DeviceView(tensor, (m, f if name == "up" else h)), device=DEVICE)
        return views


def prepare(case, seed):
    src = _Source(seed)
    if case["kind"] == "encoder":
        return {"encoder": _Encoder(case, src)}
    if case["kind"] == "rows":
        fmt, rows, dim = FORMATS[case["fmt"]], case["rows"], case["dim"]
        values, size = BLOCK[case["fmt"]]
        dense, table = src.normal(rows, dim).mul_(0.02), src.weight(case["fmt"], rows, dim)
        ids = torch.randint(0, rows, (case["lookups"],), generator=src.gen, device=DEVICE)
        out = {"quantized": torch.empty(rows * (dim // values) * size, dtype=torch.uint8, device=DEVICE),
               "dense": torch.empty(rows, dim, dtype=torch.float32, device=DEVICE),
               "looked_up": torch.empty(case["lookups"], dim, dtype=torch.float32, device=DEVICE)}
        calls = [(kernels.launchQuantizeRows, (fmt, _buf(out["quantized"]), _buf(dense), rows, dim)),
                 (kernels.launchDequantizeF32, (fmt, _lib.LAYOUT_PREPARED, _buf(out["dense"]), _buf(table), rows, dim)),
                 (kernels.launchEmbeddingLookupF32, (fmt, _lib.LAYOUT_PREPARED, _buf(out["looked_up"]), _buf(table), _buf(ids),
                                                     case["lookups"], dim, rows))]
        return {"calls": calls, "out": out, "keep": [dense, table, ids]}
    calls, out, keep = _launch_plan(case, src)
    state = {"calls": calls, "out": out, "keep": keep}
    if case.get("graph"):
        _issue(calls)  # once outside the capture, as a program warms up
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            _issue(calls)
    return state


def run(state):
    if "encoder" in state:
        return state["encoder"].step()
    if "graph" in state:
        state["graph"].replay()
    else:
        _issue(state["calls"])
    return state["out"]


def _f32(t):
    """A 64-bit value rounded once to float32, kept in 64 bits."""
    return t.float().double()


def _quantized_activations(x, block):
    """The values that an int8 activation quantizer with blocks of `block` leaves of x, in 64 bits: scale max|x| / 127, a
    reciprocal, a product and a rounding half away from zero, each as float32 defines it."""
    v = x.double().reshape(-1, block)
    peak = v.abs().amax(dim=1, keepdim=True)
    scale = torch.where(peak == 0, 1.0, _f32(peak / 127.0))
    t = _f32(v * _f32(1.0 / scale))
    return (torch.sign(t) * torch.floor(t.abs() + 0.5).clamp(max=127.0) * scale).reshape(x.shape)


def _dequantized(fmt, raw, out_dim, in_dim):
    """The values of GGUF blocks in 64 bits."""
    values, size = BLOCK[fmt]
    blocks = raw.reshape(-1, size)
    halves = blocks[:, : 4 if fmt == "q4_k" else 2].contiguous().view(torch.float16).double()
    if fmt == "q8_0":
        dense = blocks[:, 2:].contiguous().view(torch.int8).double() * halves
    elif fmt == "q4_0":
        quants = blocks[:, 2:]
        dense = (torch.cat([quants & 15, quants >> 4], dim=1).double() - 8.0) * halves
    else:
        packed, quants = blocks[:, 4:16], blocks[:, 16:].reshape(-1, 4, 32)
        low, mid, high = packed[:, 0:4], packed[:, 4:8], packed[:, 8:12]
        scales = torch.cat([low & 63, (high & 15) | (low >> 6 << 4)], dim=1).double() * halves[:, 0:1]
        minima = torch.cat([mid & 63, (high >> 4) | (mid >> 6 << 4)], dim=1).double() * halves[:, 1:2]
        nibbles = torch.stack([quants & 15, quants >> 4], dim=2).reshape(-1, 8, 32).double()
        dense = nibbles * scales[:, :, None] - minima[:, :, None]
    return dense.reshape(out_dim, in_dim)


def _product(fmt, x, raw, out_dim):
    """x times the transposed weight in 64 bits, on the activations that the library's definition of the op takes."""
    rows, in_dim = x.shape
    if fmt == "q4_k":  # 8-bit activations on a set of short inner sizes and row counts, float32 elsewhere
        counts = (1, 2, 4, 9, 50, 64, 77, 154, 197, 231, 257, 308, 514)
        quantized = 256 if out_dim >= 512 and in_dim in (512, 768, 1536, 2048, 3072) and rows in counts else 0
    else:
        quantized = 32 if out_dim >= 512 and in_dim >= 96 else 0
    values = _quantized_activations(x, quantized) if quantized else x.double()
    return values @ _dequantized(fmt, raw, out_dim, in_dim).T


def exact(case, seed):
    """What run() returns for the inputs of prepare(case, seed), by plain torch in 64 bits."""
    src, fmt, m = _Source(seed), case["fmt"], case["rows"]

    def linear(x, n):
        return _product(fmt, x, src.raw_weight(fmt, n, x.shape[1]), n)

    if case["kind"] == "linear":
        return {"y": linear(src.hidden(m, case["in_dim"]), case["out_dim"])}
    if case["kind"] == "rows":
        src.normal(m, case["dim"])  # the rows to quantize; the bytes have no 64-bit value
        table = _dequantized(fmt, src.raw_weight(fmt, m, case["dim"]), m, case["dim"])
        ids = torch.randint(0, m, (case["lookups"],), generator=src.gen, device=DEVICE)
        return {"quantized": None, "dense": table, "looked_up": table[ids]}
    h, f = case["hidden"], case["ffn"]
    if case["kind"] == "encoder":
        out = {}
        for i in range(case["layers"]):
            made = {name: (src.raw_weight(fmt, n, k), n, (src.normal(n) * 0.1).double())
                    for name, n, k in (("q", h, h), ("k", h, h), ("v", h, h), ("o", h, h), ("fc1", f, h), ("fc2", h, f))}
            x, context, residual, mid = src.hidden(m, h), src.normal(m, h), src.normal(m, h), src.hidden(m, h)
            wide = torch.nn.functional.gelu(src.normal(m, f))

            def biased(a, name, made=made):
                raw, n, bias = made[name]
                return _product(fmt, a, raw, n) + bias

            out.update({f"{i}.q": biased(x, "q"), f"{i}.k": biased(x, "k"), f"{i}.v": biased(x, "v")})
            out[f"{i}.attn"] = biased(context, "o") + residual.double()
            out[f"{i}.up"] = torch.nn.functional.gelu(biased(mid, "fc1"), approximate="tanh")
            out[f"{i}.down"] = biased(wide, "fc2") + out[f"{i}.attn"]
        return out
    layers = {name: [] for name in ("qkv", "attn", "gate", "up", "down") + (("key", "value") if case["kv"] else ())}
    for _ in range(case["layers"]):
        x = src.hidden(m, h)
        layers["qkv"].append(linear(x, case["qkv"]))
        if case["kv"]:
            layers["key"].append(linear(x, case["kv"]))
            layers["value"].append(linear(x, case["kv"]))
        layers["attn"].append(linear(src.normal(m, h), h))
        x = src.hidden(m, h)
        layers["gate"].append(linear(x, f))
        layers["up"].append(linear(x, f))
        layers["down"].append(linear(src.gated(m, f), h))
    out = {name: torch.stack(values) for name, values in layers.items()}
    if case["vocab"]:
        logits = linear(src.hidden(m, h)[-1:], case["vocab"])
        out["token"] = logits.argmax(dim=1).to(torch.int32)
    return out
