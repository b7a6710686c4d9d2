"""The calls whose speed counts, as a serving program makes them.

One OCR request is a prefill of one page's prompt (some hundred to some
thousand image and text tokens) through twelve decoder layers, then a decode
step per generated token for every page in flight. The cases are the pieces
of that work and the two whole calls, each through the engine's public entry
points on resident weights:

* ``lm_head``          final rows -> logits + argmax, or the greedy n-gram step
* ``moe_decode``       the 64-expert top-6 layer for the rows of a decode step
* ``rswa``             ring write + decode attention for the streams in flight
* ``attention``        causal prefill attention of a chunk over its prefix
* ``moe_prefill_i4``   a prefill chunk through the int4 experts
* ``linear``           a prefill projection, ``linear_int8_dynamic``
* ``layer_prefill``    one decoder layer over a prefill chunk
* ``decoder_step``     the whole decode step, twelve layers and the LM head
* ``decoder_prefill``  the whole prompt of one stream, then the first logits

Weights are seeded random codes with per-row scales of about unit gain, and of
1/16 where a projection's output is added to the residual stream (o_proj and
the down projections): a layer adds a small part of what the stream holds, as
a trained one does. Every state has its own weights, as
consecutive layers and models have.
"""

from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from franken_ocr_amd import engine
from franken_ocr_amd.device import DeviceArray, default_context

HIDDEN, INTER, EXPERTS, TOP_K = 1280, 896, 64, 6
SHARED, DENSE, VOCAB, LAYERS = 1792, 6848, 129280, 12
HEADS, HEAD_DIM, RING = engine.NUM_HEADS, engine.HEAD_DIM, engine.RING_WINDOW
DIM = HEADS * HEAD_DIM
EPS, THETA = 1e-6, 10000.0
ADDED = 0.0625  # the gain of a projection whose output is added to the residual stream
# the projections of the decoder that linear_int8_dynamic serves: (n, k)
LINEARS = {"qkv": (3 * DIM, HIDDEN), "o_proj": (HIDDEN, DIM), "dense_gate": (DENSE, HIDDEN),
           "dense_down": (HIDDEN, DENSE)}


def listed():
    return [
        # one page in flight, the first call of a user who tries it: one row through the LM head
        {"name": "lm_head_1", "kind": "lm_head", "rows": 1, "sample": False},
        # eight pages in flight, the greedy step with the no-repeat-ngram ban
        {"name": "lm_head_sample_8", "kind": "lm_head", "rows": 8, "sample": True},
        # one decode row through one MoE layer with the shared expert (the model's default routing)
        {"name": "moe_decode_1", "kind": "moe_decode", "rows": 1, "shared": True, "norm_topk": False},
        # the benchmark's headline: eight rows, renormalised gates
        {"name": "moe_decode_8", "kind": "moe_decode", "rows": 8, "shared": False, "norm_topk": True},
        # a busy server: an odd number of rows, most experts hit
        {"name": "moe_decode_29", "kind": "moe_decode", "rows": 29, "shared": True, "norm_topk": False},
        # the decode attention of eight pages with reference blocks of different lengths
        {"name": "rswa_8", "kind": "rswa", "streams": 8, "ref": 1024},
        # a page's prompt as one chunk
        {"name": "attention_1024", "kind": "attention", "rows": 1024, "start": 0},
        # a prefill chunk through a layer of int4 experts with skewed routing
        {"name": "moe_prefill_i4_512", "kind": "moe_prefill_i4", "rows": 512, "group": 32},
        # a long batch of rows through the dense layer's gate projection
        {"name": "linear_8192", "kind": "linear", "rows": 8192, "weight": "dense_gate"},
        # a prompt through one layer in chunks of 256, the last one shorter
        {"name": "layer_prefill_1000", "kind": "layer_prefill", "rows": 1000, "chunk": 256, "mlp": "moe"},
        # one token for eight pages
        {"name": "decoder_step_8", "kind": "decoder_step", "streams": 8, "ref": 1024},
        # one page's prompt in one chunk, to the first token's logits
        {"name": "decoder_prefill_1024", "kind": "decoder_prefill", "rows": 1024, "chunk": 0},
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["lm_head", "moe_decode", "rswa", "attention", "moe_prefill_i4", "linear", "layer_prefill",
                       "decoder_step", "decoder_prefill"])
    if kind == "lm_head":
        return {"kind": kind, "rows": _between(rng, 1, 32), "sample": rng.random() < 0.5}
    if kind == "moe_decode":
        return {"kind": kind, "rows": _between(rng, 1, 64), "shared": rng.random() < 0.5,
                "norm_topk": rng.random() < 0.5}
    if kind == "rswa":
        return {"kind": kind, "streams": _between(rng, 1, 24), "ref": _between(rng, 128, 2048)}
    if kind == "attention":
        rows = _between(rng, 16, 1280)
        return {"kind": kind, "rows": rows, "start": rng.choice([0, rng.randrange(1, 1025)])}
    if kind == "moe_prefill_i4":
        return {"kind": kind, "rows": _between(rng, 64, 1024), "group": rng.choice([16, 32])}
    if kind == "linear":
        return {"kind": kind, "rows": _between(rng, 16, 8192), "weight": rng.choice(sorted(LINEARS))}
    if kind == "layer_prefill":
        return {"kind": kind, "rows": _between(rng, 16, 1280), "chunk": rng.choice([0, 256]),
                "mlp": rng.choice(["moe", "moe", "dense"])}
    if kind == "decoder_step":
        return {"kind": kind, "streams": _between(rng, 1, 12), "ref": _between(rng, 128, 1024)}
    return {"kind": kind, "rows": _between(rng, 64, 1000), "chunk": rng.choice([0, 256])}


# ---- device memory ------------------------------------------------------------------


class _Memory:
    """Device memory of the engine as torch sees it; a tensor of it keeps `owner`, whose memory it is."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 2}


# torch has no arithmetic on uint32: ids are seen as int32 (they are far below 2^31)
_TYPES = {np.dtype(np.float32): "<f4", np.dtype(np.int8): "|i1", np.dtype(np.uint8): "|u1", np.dtype(np.uint32): "<i4"}


def _view(a: DeviceArray) -> torch.Tensor:
    return torch.as_tensor(_Memory(a, a.ptr, a.shape, _TYPES[a.dtype]), device="cuda")


def _region(cache: engine.RingCache, ptr, shape) -> torch.Tensor:
    return torch.as_tensor(_Memory(cache, ptr, shape, "<f4"), device="cuda")


class _Make:
    """Seeded inputs in the engine's memory."""

    def __init__(self, seed):
        self.ctx = default_context()
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))

    def put(self, t, dtype):
        a = self.ctx.empty(tuple(t.shape), dtype)
        _view(a).copy_(t)
        return a

    def normal_(self, shape, sigma=1.0):
        return torch.randn(shape, generator=self.gen, device="cuda") * sigma

    def uniform_(self, shape, lo, hi):
        return torch.rand(shape, generator=self.gen, device="cuda") * (hi - lo) + lo

    def normal(self, shape, sigma=1.0):
        return self.put(self.normal_(shape, sigma), np.float32)

    def uniform(self, shape, lo, hi):
        return self.put(self.uniform_(shape, lo, hi), np.float32)

    def codes(self, shape):
        a = self.ctx.empty(shape, np.int8)
        _view(a).copy_(torch.randint(-127, 128, shape, generator=self.gen, device="cuda", dtype=torch.int8))
        return a

    def nibbles(self, shape):
        a = self.ctx.empty(shape, np.uint8)
        _view(a).copy_(torch.randint(0, 256, shape, generator=self.gen, device="cuda", dtype=torch.uint8))
        return a

    def scales(self, shape, k, gain=1.0, deviation=73.3):
        """Per-row scales of about that gain (`deviation` is the codes' standard deviation)."""
        unit = gain / (deviation * math.sqrt(k))
        return self.uniform(shape, 0.5 * unit, 1.5 * unit)

    def weight(self, n, k, gain=1.0):
        return self.codes((n, k)), self.scales((n,), k, gain)

    def host(self, n):
        """A norm weight, which the engine takes from the host."""
        return self.uniform_((n,), 0.5, 1.5).cpu().numpy()


def _qint8(weight, ctx):
    w, s = weight
    n, k = w.shape
    return engine.QInt8(w, s, n, k, ctx=ctx)


def _moe_weights(m, shared):
    w = {"router": m.normal((EXPERTS, HIDDEN), 0.02)}
    for name, n, k, gain in (("g", INTER, HIDDEN, 1.0), ("u", INTER, HIDDEN, 1.0), ("d", HIDDEN, INTER, ADDED)):
        w["w" + name], w["s" + name] = m.codes((EXPERTS, n, k)), m.scales((EXPERTS, n), k, gain)
    if shared:
        w["shared"] = (*m.weight(SHARED, HIDDEN), *m.weight(SHARED, HIDDEN), *m.weight(HIDDEN, SHARED, ADDED))
    return w


def _moe_layer(m, w):
    layer = engine.MoeLayer(HIDDEN, INTER, EXPERTS, TOP_K, w["router"], w["wg"], w["sg"], w["wu"], w["su"], w["wd"],
                            w["sd"], ctx=m.ctx)
    if "shared" in w:
        layer.set_shared(SHARED, *w["shared"])
    return layer


def _layer_weights(m, mlp):
    w = {"ln1": m.host(HIDDEN), "ln2": m.host(HIDDEN), "qkv": m.weight(3 * DIM, HIDDEN),
         "o": m.weight(HIDDEN, DIM, ADDED)}
    if mlp == "moe":
        w["moe"] = _moe_weights(m, True)
    else:
        w["dense"] = (m.weight(DENSE, HIDDEN), m.weight(DENSE, HIDDEN), m.weight(HIDDEN, DENSE, ADDED))
    return w


def _decoder_layer(m, w):
    torch.cuda.synchronize()  # the engine reads the weights on its own stream
    if "moe" in w:
        mlp = {"moe": _moe_layer(m, w["moe"])}
    else:
        mlp = {"dense": tuple(_qint8(d, m.ctx) for d in w["dense"])}
    return engine.DecoderLayer(HIDDEN, w["ln1"], w["ln2"], _qint8(w["qkv"], m.ctx), _qint8(w["o"], m.ctx), ctx=m.ctx,
                               eps=EPS, rope_theta=THETA, **mlp)


def _lengths(ref, streams):
    """Prompt lengths of pages in flight: up to `ref` tokens, none alike."""
    return [max(1, ref - (s * 61) % max(1, ref // 2)) for s in range(streams)]


def _cache(m, lengths, capacity):
    """A ring cache in the steady state of decoding: prompts recorded, rings full."""
    cache = engine.RingCache(len(lengths), capacity, ctx=m.ctx)
    for s, n in enumerate(lengths):
        k, v = m.normal((HEADS, n, HEAD_DIM)), m.normal((HEADS, n, HEAD_DIM))
        torch.cuda.synchronize()
        cache.record_prefill(s, k, v, n)
        m.ctx.synchronize()
        regions = cache.regions(s)
        for name in ("ring_k", "ring_v"):
            _region(cache, regions[name], (HEADS, RING, HEAD_DIM)).copy_(m.normal_((HEADS, RING, HEAD_DIM)))
        cache.set_state(s, RING, (7 * s) % RING)
    return cache


def _skewed_routing(m, rows):
    """top_k distinct experts a row, Zipf(1.1) over the experts, gates that sum to one."""
    rank = torch.randperm(EXPERTS, generator=m.gen, device="cuda")
    weight = -1.1 * torch.log(torch.arange(1, EXPERTS + 1, device="cuda", dtype=torch.float32))
    noise = -torch.log(-torch.log(m.uniform_((rows, EXPERTS), 1e-6, 1.0 - 1e-6)))
    idx = rank[(weight + noise).topk(TOP_K, dim=1).indices].to(torch.int32)
    gates = m.uniform_((rows, TOP_K), 0.1, 1.0)
    return idx, gates / gates.sum(dim=1, keepdim=True)


# ---- the states ----------------------------------------------------------------------


def _lm_head_state(case, m):
    rows = case["rows"]
    w = m.weight(VOCAB, HIDDEN)
    s = {"m": m, "w": w, "q": _qint8(w, m.ctx), "x": m.normal((rows, HIDDEN)),
         "logits": m.ctx.empty((rows, VOCAB), np.float32), "tokens": m.ctx.empty((rows,), np.uint32)}
    s["out"] = (_view(s["logits"]), _view(s["tokens"]))
    if case["sample"]:
        # what the rows have generated so far: text that comes round again, so that the ban has work to do
        size, cap = 512, 1024
        ids = torch.randint(2, VOCAB, (rows, size), generator=m.gen, device="cuda")
        for r in range(rows):
            period = 40 + r
            ids[r] = ids[r, :period].repeat(-(-size // period))[:size]
        history = torch.zeros((rows, cap), dtype=torch.int32, device="cuda")
        history[:, :size] = ids.to(torch.int32)
        s["history"] = m.put(history, np.uint32)
        s["lengths"] = m.put(torch.full((rows,), size, dtype=torch.int32, device="cuda"), np.uint32)
    return s


def _moe_decode_state(case, m):
    rows = case["rows"]
    w = _moe_weights(m, case["shared"])
    torch.cuda.synchronize()
    s = {"m": m, "w": w, "layer": _moe_layer(m, w), "x": m.normal((rows, HIDDEN)),
         "y": m.ctx.empty((rows, HIDDEN), np.float32), "idx": m.ctx.empty((rows, TOP_K), np.uint32),
         "gates": m.ctx.empty((rows, TOP_K), np.float32)}
    s["out"] = tuple(_view(s[k]) for k in ("y", "idx", "gates"))
    return s


def _rswa_state(case, m):
    lengths = _lengths(case["ref"], case["streams"])
    s = {"m": m, "lengths": lengths, "cache": _cache(m, lengths, case["ref"])}
    for k in "qkv":
        s[k] = m.normal((len(lengths), DIM))
    s["y"] = m.ctx.empty((len(lengths), DIM), np.float32)
    s["out"] = _view(s["y"])
    return s


def _attention_state(case, m):
    end = case["start"] + case["rows"]
    s = {"m": m, "q": m.normal((case["rows"], DIM)), "k": m.normal((end, DIM)), "v": m.normal((end, DIM)),
         "y": m.ctx.empty((case["rows"], DIM), np.float32)}
    s["out"] = _view(s["y"])
    return s


def _moe_prefill_i4_state(case, m):
    rows, group = case["rows"], case["group"]
    w = {}
    for name, n, k in (("g", INTER, HIDDEN), ("u", INTER, HIDDEN), ("d", HIDDEN, INTER)):
        w["w" + name] = m.nibbles((EXPERTS, n, k // 2))
        w["s" + name] = m.scales((EXPERTS, n, k // group), k, deviation=4.6)
    idx, gates = _skewed_routing(m, rows)
    torch.cuda.synchronize()
    s = {"m": m, "w": w, "x": m.normal((rows, HIDDEN)), "idx": m.put(idx, np.uint32), "gates": m.put(gates, np.float32),
         "layer": engine.MoeLayerI4(HIDDEN, INTER, EXPERTS, group, w["wg"], w["sg"], w["wu"], w["su"], w["wd"],
                                    w["sd"], ctx=m.ctx),
         "y": m.ctx.empty((rows, HIDDEN), np.float32)}
    s["out"] = _view(s["y"])
    return s


def _linear_state(case, m):
    n, k = LINEARS[case["weight"]]
    w = m.weight(n, k)
    s = {"m": m, "w": w, "q": _qint8(w, m.ctx), "x": m.normal((case["rows"], k)),
         "y": m.ctx.empty((case["rows"], n), np.float32)}
    s["out"] = _view(s["y"])
    return s


def _layer_prefill_state(case, m):
    rows, chunk = case["rows"], case["chunk"] or case["rows"]
    w = _layer_weights(m, case["mlp"])
    s = {"m": m, "w": w, "layer": _decoder_layer(m, w), "embedded": m.normal((rows, HIDDEN)),
         "x": m.ctx.empty((rows, HIDDEN), np.float32), "cache": engine.RingCache(1, rows, ctx=m.ctx)}
    s["chunks"] = [(c0, s["x"].view_rows(c0, c1)) for c0, c1 in engine.prefill_chunk_bounds(rows, chunk)]
    regions = s["cache"].regions(0)
    ref = tuple(_region(s["cache"], regions[k], (HEADS, rows, HEAD_DIM)) for k in ("ref_k", "ref_v"))
    s["out"] = (_view(s["x"]), *ref)
    return s


def _decoder_state(case, m, rows, out_rows):
    layers = [_decoder_layer(m, _layer_weights(m, "moe" if i else "dense")) for i in range(LAYERS)]
    norm = m.host(HIDDEN)
    head = m.weight(VOCAB, HIDDEN)
    torch.cuda.synchronize()
    s = {"m": m, "decoder": engine.Decoder(layers, norm, _qint8(head, m.ctx), ctx=m.ctx, eps=EPS),
         "embedded": m.normal((rows, HIDDEN)), "x": m.ctx.empty((rows, HIDDEN), np.float32),
         "logits": m.ctx.empty((out_rows, VOCAB), np.float32), "tokens": m.ctx.empty((out_rows,), np.uint32)}
    s["out"] = (_view(s["x"]), _view(s["logits"]))
    return s


def _decoder_step_state(case, m):
    streams = case["streams"]
    s = _decoder_state(case, m, streams, streams)
    lengths = _lengths(case["ref"], streams)
    s["caches"] = [_cache(m, lengths, case["ref"]) for _ in range(LAYERS)]
    s["positions"] = np.array([n + RING for n in lengths], np.uint32)
    return s


def _decoder_prefill_state(case, m):
    s = _decoder_state(case, m, case["rows"], 1)
    s["caches"] = [engine.RingCache(1, case["rows"], ctx=m.ctx) for _ in range(LAYERS)]
    return s


_STATES = {"lm_head": _lm_head_state, "moe_decode": _moe_decode_state, "rswa": _rswa_state,
           "attention": _attention_state, "moe_prefill_i4": _moe_prefill_i4_state, "linear": _linear_state,
           "layer_prefill": _layer_prefill_state, "decoder_step": _decoder_step_state,
           "decoder_prefill": _decoder_prefill_state}


def prepare(case, seed):
    s = _STATES[case["kind"]](case, _Make(seed))
    s["case"] = case
    torch.cuda.synchronize()
    return s


# ---- one pass ------------------------------------------------------------------------


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "lm_head":
        if case["sample"]:
            engine.lm_head_sample_i8(s["q"], s["x"], s["tokens"], s["history"], s["lengths"], logits=s["logits"])
        else:
            engine.lm_head_i8(s["q"], s["x"], s["tokens"], s["logits"])
    elif kind == "moe_decode":
        s["layer"].decode(s["x"], s["y"], s["idx"], s["gates"], norm_topk=case["norm_topk"],
                          with_shared=case["shared"], check_route=False)
    elif kind == "rswa":
        s["cache"].step(s["q"], s["k"], s["v"], s["y"])
    elif kind == "attention":
        engine.chunk_prefill_attention(s["q"], s["k"], s["v"], HEADS, HEAD_DIM, case["start"], s["y"])
    elif kind == "moe_prefill_i4":
        s["layer"].prefill(s["x"], s["idx"], s["gates"], s["y"], check_idx=False)
    elif kind == "linear":
        engine.linear_i8_dynamic(s["q"], s["x"], s["y"])
    elif kind == "layer_prefill":
        s["x"].copy_from_device(s["embedded"])  # the rows that the layer before leaves
        for c0, x in s["chunks"]:
            s["layer"].prefill(s["cache"], 0, x, c0, check_route=False)
    elif kind == "decoder_step":
        s["x"].copy_from_device(s["embedded"])  # the embedding rows of the last tokens
        s["decoder"].step(s["caches"], s["positions"], s["x"], s["tokens"], logits=s["logits"])
    else:
        s["x"].copy_from_device(s["embedded"])
        s["decoder"].prefill(s["caches"], 0, s["x"], case["rows"], chunk=case["chunk"], token=s["tokens"],
                             logits=s["logits"])
    return s["out"]


# ---- what a pass cannot do without ---------------------------------------------------


def _linear_work(rows, n, k):
    return {"bytes": n * k + 4 * n + 4 * rows * (n + k), "flops": 2 * rows * n * k}


def _moe_work(rows, shared, group=0):
    hit = EXPERTS * (1 - (1 - TOP_K / EXPERTS) ** rows)
    values = 3 * INTER * HIDDEN
    expert = values // 2 + 4 * values // group if group else values + 4 * (2 * INTER + HIDDEN)
    total = {"bytes": hit * expert + 4 * EXPERTS * HIDDEN + 8 * rows * HIDDEN,
             "flops": 2 * rows * (TOP_K * values + EXPERTS * HIDDEN)}
    if shared:
        total["bytes"] += 3 * SHARED * HIDDEN + 4 * (2 * SHARED + HIDDEN)
        total["flops"] += 2 * rows * 3 * SHARED * HIDDEN
    return total


def _attention_work(rows, start):
    end = start + rows
    return {"bytes": 4 * DIM * (2 * rows + 2 * end), "flops": 4 * DIM * (rows * start + rows * (rows + 1) // 2)}


def _rswa_work(lengths):
    keys = sum(lengths) + RING * len(lengths)
    return {"bytes": 8 * DIM * keys + 8 * DIM * len(lengths), "flops": 4 * DIM * keys}


def _layer_work(rows, mlp, attention):
    parts = [{"bytes": 4 * DIM * HIDDEN, "flops": 8 * rows * DIM * HIDDEN}, attention]
    if mlp == "moe":
        parts.append(_moe_work(rows, True))
    else:
        parts.append({"bytes": 3 * DENSE * HIDDEN, "flops": 6 * rows * DENSE * HIDDEN})
    return _sum(parts)


def _sum(parts):
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


def work(case):
    kind = case["kind"]
    if kind == "lm_head":
        return _linear_work(case["rows"], VOCAB, HIDDEN)
    if kind == "moe_decode":
        return _moe_work(case["rows"], case["shared"])
    if kind == "rswa":
        return _rswa_work(_lengths(case["ref"], case["streams"]))
    if kind == "attention":
        return _attention_work(case["rows"], case["start"])
    if kind == "moe_prefill_i4":
        return _moe_work(case["rows"], False, case["group"])
    if kind == "linear":
        return _linear_work(case["rows"], *LINEARS[case["weight"]])
    if kind == "layer_prefill":
        return _layer_work(case["rows"], case["mlp"], _attention_work(case["rows"], 0))
    if kind == "decoder_step":
        rows, attention, out = case["streams"], _rswa_work(_lengths(case["ref"], case["streams"])), case["streams"]
    else:
        rows, attention, out = case["rows"], _attention_work(case["rows"], 0), 1
    layers = [_layer_work(rows, "moe" if i else "dense", attention) for i in range(LAYERS)]
    return _sum(layers + [_linear_work(out, VOCAB, HIDDEN)])


def tolerance(case):
    kind = case["kind"]
    if kind in ("lm_head", "linear"):
        # int8 products summed in whole numbers, two f32 multiplies: only the codes' rule could differ
        return {"rel": 1e-6}
    if kind in ("rswa", "attention"):
        # f32 dot products of 128 terms and sums over the keys, in any order
        return {"rel": 2e-6}
    if kind == "moe_decode":
        # the SwiGLU rows are quantized again: an ulp in them moves a code now and then, of one row at the least
        return {"rel": 2e-3}
    if kind == "moe_prefill_i4":
        # the same over many rows: 1.1e-4 from the result in 64 bits
        return {"rel": 5e-4, "max": 0.05}
    if kind == "layer_prefill":
        # four quantizations in a row: 3e-4 between inputs that differ by an ulp, 1.1e-2 at one value
        return {"rel": 2e-3, "max": 0.04}
    # a changed rounding in one layer moves codes in all that follow, and two rows of codes of one stream for the
    # LM head differ by 1e-2 of it: 1.3e-2 between inputs that differ by an ulp, 8.5e-2 at one value
    return {"rel": 3e-2, "max": 0.5}


# ---- the same in 64 bits -------------------------------------------------------------


def _f64(a) -> torch.Tensor:
    return (_view(a) if isinstance(a, DeviceArray) else torch.as_tensor(a, device="cuda")).double()


def _codes(x, rule):
    """The int8 codes and scales of x's rows. They are whole numbers that an f32 rule defines (the largest
    value at 127; "decode" rounds halves away from zero, "ties_even" and "dynamic" to even, and "dynamic"
    divides where the others multiply by the reciprocal), so it is that rule."""
    x = x.float()
    scale = x.abs().amax(dim=1, keepdim=True) / torch.tensor(127.0, device=x.device)
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    v = x / scale if rule == "dynamic" else x * (1.0 / scale)
    q = torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v)) if rule == "decode" else torch.round(v)
    return q.clamp(-127, 127).double(), scale.double()


def _times(x, w, s, rule):
    q, scale = _codes(x, rule)
    return (q @ _f64(w).t()) * scale * _f64(s)


def _mlp(x, weights, rule):
    wg, sg, wu, su, wd, sd = weights
    g, u = _times(x, wg, sg, rule), _times(x, wu, su, rule)
    return _times(g / (1 + torch.exp(-g)) * u, wd, sd, rule)


def _route(x, router, norm_topk):
    p = torch.softmax(x.double() @ _f64(router).t(), dim=1)
    gates, idx = p.topk(TOP_K, dim=1)
    return idx, gates / gates.sum(dim=1, keepdim=True) if norm_topk else gates


def _experts(x, idx, gates, expert, rule):
    y = torch.zeros_like(x)
    for e in range(EXPERTS):
        row, slot = (idx == e).nonzero(as_tuple=True)
        if len(row):
            y[row] += _mlp(x[row], expert(e), rule) * gates[row, slot, None]
    return y


def _moe(x, w, norm_topk, rule, shared):
    idx, gates = _route(x, w["router"], norm_topk)
    views = [_view(w[k]) for k in ("wg", "sg", "wu", "su", "wd", "sd")]
    y = _experts(x, idx, gates, lambda e: [v[e] for v in views], rule)
    return y + _mlp(x, w["shared"], rule) if shared else y, idx, gates


def _attend(q, k, v, start):
    """Causal attention of rows at `start`.. over keys [heads, end, head_dim]."""
    q = q.view(-1, HEADS, HEAD_DIM).transpose(0, 1)
    seen = torch.arange(k.shape[1], device="cuda")[None, :] <= start + torch.arange(q.shape[1], device="cuda")[:, None]
    out = []
    for h in range(HEADS):
        score = (q[h] @ k[h].t().contiguous()) / math.sqrt(HEAD_DIM)
        out.append(torch.softmax(score.masked_fill(~seen, -math.inf), dim=1) @ v[h])
    return torch.stack(out, dim=1).reshape(-1, DIM)


def _heads(x):
    return x.view(-1, HEADS, HEAD_DIM).transpose(0, 1)


def _rope(x):
    half = HEAD_DIM // 2
    freq = torch.tensor([1.0 / THETA ** (2 * i / HEAD_DIM) for i in range(half)], dtype=torch.float64, device="cuda")
    position = torch.arange(x.shape[0], device="cuda", dtype=torch.float32)
    angle = (position[:, None] * freq.float()).double()[:, None, :]  # the angle itself is an f32 product
    a, b = x.view(-1, HEADS, HEAD_DIM).split(half, dim=2)
    c, s = torch.cos(angle), torch.sin(angle)
    return torch.cat([a * c - b * s, b * c + a * s], dim=2).reshape(-1, DIM)


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPS) * _f64(w)


def _layer_exact(s):
    w, x = s["w"], _f64(s["embedded"])
    q, k, v = _times(_norm(x, w["ln1"]), *w["qkv"], "dynamic").split(DIM, dim=1)
    k, v = _heads(_rope(k)), _heads(v)
    x = x + _times(_attend(_rope(q), k, v, 0), *w["o"], "dynamic")
    n = _norm(x, w["ln2"])
    if "moe" in w:
        y = _moe(n, w["moe"], False, "dynamic", True)[0]
    else:
        y = _mlp(n, [a for pair in w["dense"] for a in pair], "dynamic")
    return x + y, k, v


def _banned(history, size, ngram, window):
    """The ids that would end an n-gram of the last `window` tokens a second time."""
    seq = history[:size]
    last = seq[size - (ngram - 1):]
    return {seq[i + ngram - 1] for i in range(max(0, size - window), size - ngram + 1) if seq[i:i + ngram - 1] == last}


def _rswa_exact(s):
    out = []
    q, k, v = (_f64(s[n]).view(-1, HEADS, HEAD_DIM) for n in "qkv")
    for i, n in enumerate(s["lengths"]):
        r = s["cache"].regions(i)
        slot = s["cache"].state(i)[2]
        ref = [_region(s["cache"], r[name], (HEADS, s["case"]["ref"], HEAD_DIM))[:, :n].double()
               for name in ("ref_k", "ref_v")]
        ring = [_region(s["cache"], r[name], (HEADS, RING, HEAD_DIM)).double() for name in ("ring_k", "ring_v")]
        ring[0][:, slot], ring[1][:, slot] = k[i], v[i]  # the step's own token takes the oldest one's place
        keys, values = (torch.cat([a, b], dim=1) for a, b in zip(ref, ring))
        p = torch.softmax((keys @ q[i][:, :, None]).squeeze(2) / math.sqrt(HEAD_DIM), dim=1)
        out.append((p[:, None, :] @ values).reshape(DIM))
    return torch.stack(out)



def _nibbles(w):
    """[n, k/2] packed codes -> [n, k], the low nibble first."""
    w = w.to(torch.int16)
    lo, hi = ((w & 15) ^ 8) - 8, ((w >> 4) ^ 8) - 8
    return torch.stack([lo, hi], dim=2).view(w.shape[0], -1).double()


def _moe_i4_exact(s, group):
    x, idx, gates = _f64(s["x"]), _view(s["idx"]), _f64(s["gates"])

    def times(q, scale, name, e):
        w = _nibbles(_view(s["w"]["w" + name])[e])
        return (q @ (w * _f64(_view(s["w"]["s" + name])[e]).repeat_interleave(group, dim=1)).t()) * scale

    y = torch.zeros_like(x)
    for e in range(EXPERTS):
        row, slot = (idx == e).nonzero(as_tuple=True)
        if len(row):
            q = _codes(x[row], "ties_even")
            g, u = times(*q, "g", e), times(*q, "u", e)
            a = _codes(g / (1 + torch.exp(-g)) * u, "ties_even")
            y[row] += times(*a, "d", e) * gates[row, slot, None]
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decoder_step", "decoder_prefill"):
        # twelve layers of rounding to int8 codes and of choosing experts: two correct results part at the first
        # code that falls the other way, and there is no value that both are near in the sense of 64 bits
        return None
    s = prepare(case, seed)
    if kind == "lm_head":
        logits = _times(_f64(s["x"]), *s["w"], "decode")
        if case["sample"]:
            size = _view(s["lengths"]).tolist()
            for r, history in enumerate(_view(s["history"]).tolist()):
                for t in _banned(history, size[r], engine.DEFAULT_NO_REPEAT_NGRAM_SIZE, engine.NGRAM_WINDOW_SINGLE):
                    logits[r, t] = -math.inf
        return logits, None
    if kind == "moe_decode":
        y, _, gates = _moe(_f64(s["x"]), s["w"], case["norm_topk"], "decode", case["shared"])
        return y, None, gates
    if kind == "rswa":
        return _rswa_exact(s)
    if kind == "attention":
        return _attend(_f64(s["q"]), _heads(_f64(s["k"])), _heads(_f64(s["v"])), case["start"])
    if kind == "moe_prefill_i4":
        return _moe_i4_exact(s, case["group"])
    if kind == "linear":
        return _times(_f64(s["x"]), *s["w"], "dynamic")
    return _layer_exact(s)
