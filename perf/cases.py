"""The work by which this library's speed is judged: quantized decode matvecs, whole decode steps, and quantized
prefill matmuls, called the way a host program calls them (openagents_amd.backend, openagents_amd.decode).

A case is one of five kinds:

  matvec       one psn_qmatvec launched eagerly
  projections  the four projection launches of `layers` decoder layers (q|k|v, o, gate|up, down) at batch 1..8,
               replayed from a graph or launched one by one from the host
  token        one decode step of a llama-shaped model at a given context: a graph replay, or what greedy decoding does
               per token (embedding row up, every launch from the host, logits down)
  prefill      the seven projections of one layer for M tokens at once
  packed       the same on weights dequantized once beforehand (psn_prefill_pack)

Weights are rows of N(0, 0.02) quantized by the library's own host quantizers.  A pool of such rows is quantized per
row length and every matrix takes its rows from it in an order of its own, so that a model is made in a second; a
row's bytes are those a checkpoint's conversion would hold.  Activations are N(0, 1), KV caches fp16 N(0, 1).
Everything is sized by layer so that a pass reads its weights from HBM and not from a cache.
"""
import ctypes
import math

import numpy as np
import torch

from openagents_amd import decode, quantize
from openagents_amd._ffi import ACT_F32, ACT_Q8, Q4_0, Q4_K, Q5_K, Q6_K, Q8_0
from openagents_amd.backend import DeviceBuffer, HipBackend, QuantizedTensor, row_bytes

FORMATS = {"q4_0": Q4_0, "q8_0": Q8_0, "q4_K": Q4_K, "q5_K": Q5_K, "q6_K": Q6_K}
HEAD = 128
POOL_ROWS = 512

# the 8B shape of the repository's benchmark, and its 70B-class layer
S8B = {"hidden": 4096, "kv_heads": 8, "ffn": 14336}
S70B = {"hidden": 8192, "kv_heads": 8, "ffn": 28672}


def listed():
    return [
        # the smallest call a host program makes: one 4096 x 4096 matrix against one vector, launched on its own
        {"name": "matvec_q8_0_4096", "kind": "matvec", "fmt": "q8_0", "n": 4096, "k": 4096, "batch": 1, "scheme": "q8"},
        # single-sequence decode, projections only: the benchmark's headline workload (eight of its layers)
        {"name": "projections_q4_0_b1", "kind": "projections", "fmt": "q4_0", "batch": 1, "layers": 8, "scheme": "q8", "graph": True, **S8B},
        # eight sequences decoded together, the format of the 8B decode model
        {"name": "projections_q4_K_b8", "kind": "projections", "fmt": "q4_K", "batch": 8, "layers": 4, "scheme": "q8", "graph": True, **S8B},
        # four sequences, 8-bit weights, 70B-class layer, a host loop without a graph
        {"name": "projections_q8_0_b4", "kind": "projections", "fmt": "q8_0", "batch": 4, "layers": 1, "scheme": "q8", "graph": False, **S70B},
        # one token of the 8B shape at 2048 positions, graph replay (eight of its 32 layers and the whole LM head)
        {"name": "token_8b_2k", "kind": "token", "fmt": "q4_K", "fmt2": "q4_K", "layers": 8, "vocab": 128256, "ctx": 2048, "graph": True, **S8B},
        # the same from a greedy host loop, early in a conversation; value and down projections of another format, as
        # the K-quant mixes of model files have them
        {"name": "token_8b_host_loop", "kind": "token", "fmt": "q4_K", "fmt2": "q6_K", "layers": 8, "vocab": 128256, "ctx": 301, "graph": False, **S8B},
        # far into a long document: attention over 24 000 positions
        {"name": "token_long_context", "kind": "token", "fmt": "q8_0", "fmt2": "q8_0", "layers": 4, "vocab": 32000, "ctx": 24000, "graph": True, **S8B},
        # a short question
        {"name": "prefill_33", "kind": "prefill", "fmt": "q4_K", "m": 33, **S8B},
        # an ordinary prompt of odd length
        {"name": "prefill_203", "kind": "prefill", "fmt": "q5_K", "m": 203, **S8B},
        # one chunk of chunked prefill
        {"name": "prefill_512", "kind": "prefill", "fmt": "q4_0", "m": 512, **S8B},
        # a long prompt
        {"name": "prefill_2048", "kind": "prefill", "fmt": "q4_K", "m": 2048, **S8B},
        # the longest, on a server that keeps the dequantized weights beside the quantized ones
        {"name": "packed_4001", "kind": "packed", "fmt": "q6_K", "m": 4001, **S8B},
    ]


LARGEST = 2.0 * 4001 * 218103808            # operations of the largest listed case


def draw(rng):
    def spread(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    def layer():
        hidden = 256 * max(4, round(spread(1024, 8192) / 256))
        heads = hidden // HEAD
        group = rng.choice([g for g in (1, 2, 4, 8) if heads % g == 0])
        return {"hidden": hidden, "kv_heads": heads // group, "ffn": 256 * round(hidden * rng.uniform(2.5, 3.6) / 256)}

    kind = rng.choice(["matvec", "projections", "projections", "projections", "token", "token", "prefill", "prefill", "prefill", "packed"])
    fmt = rng.choice(sorted(FORMATS))
    if kind == "matvec":
        return {"kind": kind, "fmt": fmt, "n": round(spread(200, 40000)), "k": 256 * round(spread(256, 16384) / 256), "batch": rng.choice([1, 1, 1, 2, 3, 5, 8]),
                "scheme": rng.choice(["q8", "q8", "q8", "f32"])}
    s = layer()
    if kind == "projections":
        return {"kind": kind, "fmt": fmt, "batch": rng.randint(1, 8), "layers": max(1, min(8, round(9e8 / params(s)))),
                "scheme": rng.choice(["q8", "q8", "q8", "q8", "f32"]), "graph": rng.random() < 0.7, **s}
    if kind == "token":
        return {"kind": kind, "fmt": fmt, "fmt2": rng.choice([fmt, "q6_K"]), "layers": max(2, min(8, round(1.7e9 / params(s)))), "vocab": round(spread(8000, 128256)),
                "ctx": round(spread(16, 32000)), "graph": rng.random() < 0.6, **s}
    m = round(spread(1 if kind == "prefill" else 64, 4096))
    while 2.0 * m * params(s) > LARGEST:
        m = m * 3 // 4
    return {"kind": kind, "fmt": fmt, "m": m, **s}


# ---------------------------------------------------------------------- sizes

def matrices(c):
    """(name, rows, columns) of a layer's seven projections"""
    h, f, kv = c["hidden"], c["ffn"], c["kv_heads"] * HEAD
    return [("wq", h, h), ("wk", kv, h), ("wv", kv, h), ("wo", h, h), ("w_gate", f, h), ("w_up", f, h), ("w_down", h, f)]


def params(c):
    return sum(n * k for _, n, k in matrices(c))


def layer_formats(c):
    """the format of each projection: fmt2 (where there is one) for the value and down projections"""
    second = c.get("fmt2", c["fmt"])
    return {name: second if name in ("wv", "w_down") else c["fmt"] for name, _, _ in matrices(c)}


# ---------------------------------------------------------------------- device side

_be = None


def backend():
    """One backend and one stream, as a program keeps them; its workspace is sized once, before any graph is captured."""
    global _be
    if _be is None:
        _be = HipBackend(0)
        _be.reserve(1 << 16, 8)
        _be.reserve_prefill(32768, 8192)
    return _be


class _Memory:
    def __init__(self, buf, interface):
        self.buf = buf
        self.__cuda_array_interface__ = interface


def view(buf, dtype, shape):
    """A torch tensor over the memory of a DeviceBuffer, which it keeps alive (torch holds the object it was made from).
    psn_buf is {context, device address, bytes}; the third field is checked against psn_buf_size before the second is believed."""
    fields = (ctypes.c_uint64 * 3).from_address(buf.handle.value)
    assert fields[2] == buf.nbytes == _be.lib.psn_buf_size(buf.handle), "psn_buf holds something else"
    code = {torch.float32: "<f4", torch.float16: "<f2", torch.uint8: "|u1"}[dtype]

    return torch.as_tensor(_Memory(buf, {"shape": tuple(shape), "typestr": code, "data": (fields[1], False), "version": 2}), device="cuda")


def forget_misses():
    """The library looks a kernel up in one code object after the other when it is first launched, and HIP remembers the
    misses as this thread's last error, which torch would report as its own next launch's: cleared here."""
    _be.lib.hipGetLastError()


class Made:
    """What one state owns; a graph has to be destroyed by hand."""

    def __init__(self, seed):
        self.be = backend()
        self.seed = seed
        self.rng = np.random.default_rng([seed, 20])
        self.gen = torch.Generator(device="cuda").manual_seed(seed * 7919 + 1)
        self.pools = {}
        self.graph = None

    def __del__(self):
        if getattr(self, "graph", None) is not None:
            self.be.sync()
            self.be.destroy_graph(self.graph)

    def capture(self, enqueue):
        self.be.begin_capture()
        enqueue()
        self.graph = self.be.end_capture()
        forget_misses()

    def weight(self, fmt, n, k):
        if (fmt, k) not in self.pools:
            x = self.rng.standard_normal((POOL_ROWS, k), dtype=np.float32) * np.float32(0.02)
            self.pools[fmt, k] = torch.from_numpy(quantize.quantize(FORMATS[fmt], x, 8)).cuda()
        buf = self.be.alloc(n * row_bytes(FORMATS[fmt], k))
        pick = torch.randint(POOL_ROWS, (n,), generator=self.gen, device="cuda")
        out = view(buf, torch.uint8, (n, buf.nbytes // n))
        for at in range(0, n, 16384):
            out[at:at + 16384] = self.pools[fmt, k][pick[at:at + 16384]]
        return QuantizedTensor(buf, FORMATS[fmt], n, k)

    def normal(self, shape, dtype=torch.float32, scale=1.0):
        buf = self.be.alloc(math.prod(shape) * (4 if dtype == torch.float32 else 2))
        view(buf, dtype, shape).copy_(torch.randn(shape, generator=self.gen, device="cuda") * scale)
        return buf

    def output(self, *shape):
        """A result buffer and its tensor; what it holds before the call is no result."""
        buf = self.be.alloc(math.prod(shape) * 4)
        t = view(buf, torch.float32, shape)
        t.fill_(float("nan"))
        return buf, t

    def layer(self, c):
        kinds = layer_formats(c)
        return {name: self.weight(kinds[name], n, k) for name, n, k in matrices(c)}


def prepare(case, seed):
    made = Made(seed)
    state = {"matvec": prepare_matvec, "projections": prepare_projections, "token": prepare_token, "prefill": prepare_prefill, "packed": prepare_prefill}[case["kind"]](case, made)
    made.pools = {}
    torch.cuda.synchronize()
    return state


def run(state):
    outs = state[0](*state[1:])
    forget_misses()
    return outs


# ---------------------------------------------------------------------- matvec, projections

def prepare_matvec(c, made):
    w, x = made.weight(c["fmt"], c["n"], c["k"]), made.normal((c["batch"], c["k"]))
    y, out = made.output(c["batch"], c["n"])
    return run_matvec, made, w, x, y, c["batch"], ACT_F32 if c["scheme"] == "f32" else ACT_Q8, out


def run_matvec(made, w, x, y, batch, scheme, out):
    made.be.quantized_matvec(w, x, y, batch, scheme)
    return out


def prepare_projections(c, made):
    b, scheme = c["batch"], ACT_F32 if c["scheme"] == "f32" else ACT_Q8
    x, attn, act = made.normal((b, c["hidden"])), made.normal((b, c["hidden"])), made.normal((b, c["ffn"]))
    launches, outs = [], []
    for _ in range(c["layers"]):
        w = made.layer(c)
        for names, src in ((("wq", "wk", "wv"), x), (("wo",), attn), (("w_gate", "w_up"), x), (("w_down",), act)):
            ys = [made.output(b, w[name].n) for name in names]
            launches.append(([w[name] for name in names], src, [y for y, _ in ys]))
            outs += [t for _, t in ys]

    def enqueue():
        for ws, src, ys in launches:
            made.be.quantized_matvec_multi(ws, src, ys, b, scheme)

    if c["graph"]:
        made.capture(enqueue)
    return run_graph if c["graph"] else run_eager, made, enqueue, outs


def run_graph(made, enqueue, outs):
    made.be.launch_graph(made.graph)
    return outs


def run_eager(made, enqueue, outs):
    enqueue()
    return outs


# ---------------------------------------------------------------------- one token

def prepare_token(c, made):
    be = made.be
    shape = decode.LlamaShape(hidden=c["hidden"], n_heads=c["hidden"] // HEAD, n_kv_heads=c["kv_heads"], head_dim=HEAD, ffn=c["ffn"], vocab=c["vocab"], n_layers=c["layers"])

    def norm():
        buf = be.alloc(c["hidden"] * 4)
        view(buf, torch.float32, (c["hidden"],)).copy_(1.0 + 0.1 * torch.randn(c["hidden"], generator=made.gen, device="cuda"))
        return buf

    layers = [decode.LayerWeights(**made.layer(c), attn_norm=norm(), ffn_norm=norm()) for _ in range(c["layers"])]
    step = decode.DecodeStep(be, shape, decode.ModelWeights(layers, norm(), made.weight("q6_K", c["vocab"], c["hidden"])), c["ctx"])
    caches = []
    for buf in (b for pair in zip(step.k_cache, step.v_cache) for b in pair):
        t = view(buf, torch.float16, (c["ctx"], shape.kv_dim))
        t.copy_(torch.randn(t.shape, generator=made.gen, device="cuda", dtype=torch.float16))
        caches.append(t)
    row = made.rng.standard_normal(c["hidden"], dtype=np.float32)
    pos = c["ctx"] - 1
    if not c["graph"]:
        return run_token_host_loop, made, step, row, pos, caches
    # the step overwrites its residual stream: every replay is preceded by a copy of the embedding row, as a table on the device would supply it
    src = be.upload(row)
    made.capture(lambda: step.enqueue(pos))
    return run_token_graph, made, step, src, [view(step.logits, torch.float32, (c["vocab"],)), *caches]


def run_token_graph(made, step, src, outs):
    made.be.copy(step.x, src, src.nbytes)
    made.be.launch_graph(made.graph)
    return outs


def run_token_host_loop(made, step, row, pos, caches):
    step.x.upload(row)
    step.enqueue(pos)
    return [step.logits.download(np.float32, (step.shape.vocab,)), *caches]


# ---------------------------------------------------------------------- prefill

def prepare_prefill(c, made):
    m = c["m"]
    x = {c["hidden"]: made.normal((m, c["hidden"]), torch.float16), c["ffn"]: made.normal((m, c["ffn"]), torch.float16)}
    calls, outs = [], []
    for name, w in made.layer(c).items():
        y, t = made.output(m, w.n)
        packed = made.be.pack_for_prefill(w) if c["kind"] == "packed" else None
        forget_misses()
        calls.append((w, packed, x[w.k], y))
        outs.append(t)
    return run_packed if c["kind"] == "packed" else run_prefill, made, calls, m, outs


def run_prefill(made, calls, m, outs):
    for w, _, x, y in calls:
        made.be.quantized_matmul(w, x, y, m)
    return outs


def run_packed(made, calls, m, outs):
    for w, packed, x, y in calls:
        made.be.quantized_matmul_packed(packed, x, y, m, w.n, w.k)
    return outs


# ---------------------------------------------------------------------- what a pass cannot do without

def work(c):
    if c["kind"] == "matvec":
        return {"bytes": c["n"] * row_bytes(FORMATS[c["fmt"]], c["k"]) + 4 * c["batch"] * (c["n"] + c["k"]), "flops": 2 * c["batch"] * c["n"] * c["k"]}
    kinds, mats = layer_formats(c), matrices(c)
    weights = sum(n * row_bytes(FORMATS[kinds[name]], k) for name, n, k in mats)
    rows = sum(n for _, n, _ in mats)
    if c["kind"] == "projections":
        b = c["batch"]
        return {"bytes": c["layers"] * (weights + 4 * b * rows) + 4 * b * (2 * c["hidden"] + c["ffn"]), "flops": 2 * b * c["layers"] * params(c)}
    if c["kind"] == "token":
        kv = c["kv_heads"] * HEAD
        head = c["vocab"] * row_bytes(Q6_K, c["hidden"]) + 4 * c["vocab"]
        cache = 2 * c["ctx"] * kv * 2
        return {"bytes": c["layers"] * (weights + cache + 8 * c["hidden"]) + head,
                "flops": c["layers"] * (2 * params(c) + 4 * c["ctx"] * c["hidden"]) + 2 * c["vocab"] * c["hidden"]}
    m = c["m"]
    if c["kind"] == "packed":
        weights = 2 * params(c)
    return {"bytes": weights + 2 * m * (c["hidden"] + c["ffn"]) + 4 * m * rows, "flops": 2 * m * params(c)}


def tolerance(c):
    # int8 dot products are exact and fp16 products are exact in fp32: what differs is the order of fp32 sums.  Against sums
    # in float64 the prefill results are off by 4e-7 (largest 3e-6) at K = 14336.
    if c["kind"] != "token":
        return {"rel": 2e-6, "max": 2e-5}
    # A decode step quantizes its activations to int8 at every projection: a last-bit difference in a norm's or the
    # attention's sum moves a value that sits on a rounding boundary, and the layers behind it pass the difference on.
    # The same step with its norms summed and its activations quantized in launches of their own differs by 5e-3 in the
    # logits (largest 1.5e-2) where one such value moved, 2e-7 where none did.
    return {"rel": 0.02, "max": 0.1}
