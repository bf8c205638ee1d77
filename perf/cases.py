"""Workloads of the nano-vllm-rs kernels as a serving program runs them.

Shapes are those of bench.py and the runner (host/model.cpp): hidden 1024,
16 q heads over 8 KV heads of 128, intermediate 3072, vocabulary 151936, 28
layers, KV blocks of 256 slots, at most 1024 prompt tokens a forward and 4096
tokens of context. Weights, activations and caches are random; activations
that a norm precedes are unit normal, projections keep their input's scale,
and those that end in the residual stream are scaled down by the depth, as
initialisations of deep decoders do.

Each case goes through nvr.Gpu. Decode work is captured once as a graph and
replayed, as the runner does for each decode batch size; prompt work, whose
shapes change with each batch, is launched call by call.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-rs_amd"))

import nvr  # noqa: E402

H, I, QH, KVH, D, V, LAYERS = 1024, 3072, 16, 8, 128, 151936, 28
HEADS = QH + 2 * KVH
EPS, THETA, MAX_CTX, BS = 1e-6, 1e6, 4096, 256
FUSED_ROWS = 16  # rows up to which the runner takes the fused norm + GEMM launches

_gpu = None


def gpu():
    global _gpu
    if _gpu is None:
        torch.cuda.init()
        _gpu = nvr.Gpu(0)
    return _gpu


# ------------------------------------------------------------------- cases --
def listed():
    return [
        # One user, one decoder layer of a decode step: launches and latency are all there is.
        {"name": "decode_layer_1", "kind": "decode", "rows": 1, "context": 200, "layers": 1, "head": False},
        # The throughput benchmark's decode step: 8 sequences after prompts of 128 tokens, to the logits.
        {"name": "decode_step_8", "kind": "decode", "rows": 8, "context": 250, "layers": LAYERS, "head": True},
        # A full batch of the runner's default 32 sequences, a thousand tokens in.
        {"name": "decode_layer_32", "kind": "decode", "rows": 32, "context": 1024, "layers": 1, "head": False},
        # Attention of a small decode batch at a long context, over a few layers' caches.
        {"name": "attn_decode_8x1024", "kind": "attn_decode", "rows": 8, "context": 1024, "layers": 4},
        # Attention of a large decode batch at the longest context: the KV cache streams from HBM.
        {"name": "attn_decode_64x4096", "kind": "attn_decode", "rows": 64, "context": 4096, "layers": 1},
        # Attention over the throughput benchmark's prefill: 8 short prompts, unequal lengths, 1024 rows in all.
        {"name": "attn_prefill_8", "kind": "attn_prefill", "prompts": 8, "tokens": 1024, "start": 0},
        # One odd-length prompt that fills the forward.
        {"name": "attn_prefill_1x1021", "kind": "attn_prefill", "prompts": 1, "tokens": 1021, "start": 0},
        # The last chunk of the longest prompt.
        {"name": "attn_prefill_chunk", "kind": "attn_prefill", "prompts": 1, "tokens": 1024, "start": 3072},
        # One whole decoder layer over a full prefill forward.
        {"name": "prefill_layer_1024", "kind": "prefill", "prompts": 8, "tokens": 1024, "layers": 1},
        # The fused per-layer kernels alone at the bench's 8192 tokens.
        {"name": "stream_8192", "kind": "stream", "tokens": 8192},
        # Final norm of the sampled rows and the tied head for 32 sequences.
        {"name": "head_32", "kind": "head", "rows": 1024, "samples": 32},
        # Sampling of the bench's largest batch, half greedy and half at T = 0.6.
        {"name": "sample_256", "kind": "sample", "rows": 256},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "attn_decode", "attn_decode", "attn_prefill", "attn_prefill", "attn_prefill",
                       "prefill", "prefill", "stream", "head", "sample"])
    if kind == "decode":
        return {"kind": kind, "rows": rng.randint(1, 32), "context": _log_int(rng, 20, 1024),
                "layers": rng.randint(1, 4), "head": rng.random() < 0.3}
    if kind == "attn_decode":
        rows = _log_int(rng, 1, 64)
        return {"kind": kind, "rows": rows, "context": _log_int(rng, 64, 4096), "layers": rng.randint(1, 4) if rows <= 16 else 1}
    if kind == "attn_prefill":
        tokens = _log_int(rng, 64, 1024)
        start = rng.choice([0, 0, rng.randint(1, MAX_CTX - tokens)])
        return {"kind": kind, "prompts": 1 if start else rng.randint(1, min(8, tokens // 16)), "tokens": tokens,
                "start": start}
    if kind == "prefill":
        tokens = _log_int(rng, 64, 1024)
        return {"kind": kind, "prompts": rng.randint(1, min(8, tokens // 16)), "tokens": tokens, "layers": 1}
    if kind == "stream":
        return {"kind": kind, "tokens": _log_int(rng, 256, 8192)}
    if kind == "head":
        samples = rng.randint(1, 32)
        return {"kind": kind, "rows": rng.randint(samples, 1024), "samples": samples}
    return {"kind": "sample", "rows": _log_int(rng, 1, 256)}


# ------------------------------------------------------------ device plumbing --
class _Memory:
    """A device buffer in the form torch takes views of."""

    def __init__(self, buffer, typestr, shape):
        self.buffer = buffer
        self.__cuda_array_interface__ = {"data": (buffer.ptr, False), "typestr": typestr, "shape": tuple(shape),
                                         "strides": None, "version": 3}


_KINDS = {torch.bfloat16: ("<i2", 2), torch.int32: ("<i4", 4), torch.int64: ("<i8", 8), torch.float32: ("<f4", 4)}


def _view(buffer, shape, dtype=torch.bfloat16):
    t = torch.as_tensor(_Memory(buffer, _KINDS[dtype][0], shape), device="cuda")
    return t.view(dtype) if dtype == torch.bfloat16 else t


def _empty(shape, dtype=torch.bfloat16):
    return gpu().alloc(math.prod(shape) * _KINDS[dtype][1])


def _put(values):
    """A buffer of the library with these values."""
    buffer = _empty(values.shape, values.dtype)
    gpu().sync()
    _view(buffer, values.shape, values.dtype).copy_(values)
    return buffer


class _Inputs:
    """Random tensors on the GPU from one seed, made in a fixed order."""

    def __init__(self, seed):
        self.seed, self.g = int(seed), torch.Generator(device="cuda")
        self.g.manual_seed(self.seed)
        self.r = random.Random(self.seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        return (torch.randn(shape, generator=self.g, device="cuda") * std + mean).to(torch.bfloat16)

    def weight(self, n, k, gain=1.0):
        return self.normal(n, k, std=gain * k ** -0.5)

    def ints(self, low, high, *shape):
        return torch.randint(low, high, shape, generator=self.g, device="cuda", dtype=torch.int32)


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _sequences(case):
    """(first position, rows) of each sequence of the case's batch."""
    if case["kind"] in ("attn_prefill", "prefill"):
        share = [2 + i % 3 for i in range(case["prompts"])]
        ends = [case["tokens"] * sum(share[:i + 1]) // sum(share) for i in range(len(share))]
        return [(case.get("start", 0), b - a) for a, b in zip([0] + ends, ends)]
    return [(case["context"] - 1 - (r * 37) % max(1, case["context"] // 2), 1) for r in range(case["rows"])]


class _Batch:
    """Positions, sequence ids, slots and block tables of a batch over a shuffled block pool."""

    def __init__(self, case, x):
        seqs = _sequences(case)
        need = [-(-(first + rows) // BS) for first, rows in seqs]
        self.stride = MAX_CTX // BS
        self.blocks = sum(need) + 1
        ids = list(range(self.blocks))
        x.r.shuffle(ids)
        self.tables_list, at = [], 0
        for n in need:
            self.tables_list.append(ids[at:at + n] + [-1] * (self.stride - n))
            at += n
        pos, sid, slot = [], [], []
        for s, (first, rows) in enumerate(seqs):
            for p in range(first, first + rows):
                pos.append(p)
                sid.append(s)
                slot.append(self.tables_list[s][p // BS] * BS + p % BS)
        self.rows, self.seqs, self.count = len(pos), seqs, len(seqs)
        self.last_list = [sum(n for _, n in seqs[:s + 1]) - 1 for s in range(len(seqs))]
        self.pos_list, self.sid_list, self.slot_list = pos, sid, slot

    def upload(self):
        self.positions, self.ids, self.slots = (_put(_i32(v)) for v in (self.pos_list, self.sid_list, self.slot_list))
        self.tables, self.last = _put(_i32(self.tables_list)), _put(_i32(self.last_list))
        return self


def _rope_table():
    buffer = _empty((MAX_CTX, D), torch.float32)
    gpu().rope_cache(buffer, MAX_CTX, D, THETA)
    return buffer


# The values of a case, by seed, as torch tensors: prepare() puts them into the library's buffers and
# exact() computes with them.
def _layer_values(x):
    deep = (2 * LAYERS) ** -0.5
    return {"input_norm": x.normal(H, std=0.1, mean=1.0), "qkv": x.weight(HEADS * D, H),
            "q_norm": x.normal(D, std=0.1, mean=1.0), "k_norm": x.normal(D, std=0.1, mean=1.0),
            "o_proj": x.weight(H, QH * D, deep), "post_norm": x.normal(H, std=0.1, mean=1.0),
            "gate_up": x.weight(2 * I, H), "down": x.weight(H, I, deep)}


def _tiled(gate_up):
    """gate_up's rows in the order that rms_gemm_silu takes: 8 gate rows, then their 8 up rows."""
    return torch.cat([gate_up[:I].view(-1, 8, H), gate_up[I:].view(-1, 8, H)], 1).reshape(2 * I, H).contiguous()


# ----------------------------------------------------------------- prepare --
def prepare(case, seed):
    x = _Inputs(seed)
    state = _PREPARE[case["kind"]](dict(case), x)
    torch.cuda.synchronize()
    gpu().sync()
    if state.get("steps") is not None and case["kind"] in ("decode", "attn_decode"):
        state["steps"]()  # first use of each GEMM shape stays outside the capture
        gpu().sync()
        state["graph"] = gpu().capture(state["steps"])
    return state


def _prepare_model(case, x):
    """The decoder layers over a batch, in the runner's launch order (host/model.cpp)."""
    g, b, layers, decode = gpu(), _Batch(case, x).upload(), case["layers"], case["kind"] == "decode"
    n, head = b.rows, case.get("head", False)
    fused = decode and n <= FUSED_ROWS
    table_rows = V if head else 4096
    table = x.normal(table_rows, H)
    tokens = x.ints(0, table_rows, n)
    kc, vc = _put(x.normal(layers, b.blocks, BS, KVH, D)), _put(x.normal(layers, b.blocks, BS, KVH, D))
    w = []
    for _ in range(layers):
        values = _layer_values(x)
        if fused:
            values["gate_up"] = _tiled(values["gate_up"])
        w.append({k: _put(t) for k, t in values.items()})
        torch.cuda.synchronize()
    final = _put(x.normal(H, std=0.1, mean=1.0))
    table, tokens, rope = _put(table), _put(tokens), _rope_table()
    residual, other, hidden, normed, gathered = (_empty((n, H)) for _ in range(5))
    qkv, query, attn = _empty((n, HEADS * D)), _empty((n, QH * D)), _empty((n, QH * D))
    gate_up, act = _empty((n, 2 * I)), _empty((n, I))
    logits = _empty((b.count, V)) if head else None
    span = b.blocks * BS * KVH * D * 2
    kcs, vcs = [kc.slice(i * span, span) for i in range(layers)], [vc.slice(i * span, span) for i in range(layers)]
    # With fused norms each add-norm reads one residual buffer and writes the other: two a layer, one in the first.
    out_residual = residual if not fused or (2 * layers - 1) % 2 == 0 else other

    def steps():
        now, nxt = residual, other
        g.embedding(tokens, table, now, n, H, table_rows)
        for i, l in enumerate(w):
            if fused and i == 0:
                g.rms_gemm(now, None, None, l["input_norm"], l["qkv"], qkv, normed, n, HEADS * D, H, EPS)
            elif fused:
                g.rms_gemm(hidden, now, nxt, l["input_norm"], l["qkv"], qkv, normed, n, HEADS * D, H, EPS)
                now, nxt = nxt, now
            else:
                if i == 0:
                    g.rms_norm(now, l["input_norm"], normed, n, H, EPS)
                else:
                    g.add_rms_norm(hidden, now, l["input_norm"], normed, n, H, EPS)
                g.gemm(normed, l["qkv"], qkv, n, HEADS * D, H)
            if decode:
                g.attention_qkv_rope(qkv, l["q_norm"], l["k_norm"], b.positions, b.slots, kcs[i], vcs[i], b.ids,
                                     b.tables, attn, n, QH, KVH, D, BS, b.blocks, b.stride, b.count, MAX_CTX, EPS,
                                     rope, MAX_CTX)
            else:
                g.qkv_rope_cached(qkv, l["q_norm"], l["k_norm"], b.positions, b.slots, query, kcs[i], vcs[i], n, QH,
                                  KVH, D, BS, b.blocks, EPS, rope, MAX_CTX)
                g.paged_attention(query, kcs[i], vcs[i], b.positions, b.ids, b.tables, attn, n, QH, KVH, D, BS,
                                  b.blocks, b.stride, b.count, MAX_CTX)
            if fused:
                g.gemm_rows(attn, l["o_proj"], hidden, n, H, QH * D)
                g.rms_gemm_silu(hidden, now, nxt, l["post_norm"], l["gate_up"], gate_up, act, normed, n, I, H, EPS)
                now, nxt = nxt, now
                g.gemm_rows(act, l["down"], hidden, n, H, I)
            else:
                g.gemm(attn, l["o_proj"], hidden, n, H, QH * D)
                g.add_rms_norm(hidden, now, l["post_norm"], normed, n, H, EPS)
                g.gemm(normed, l["gate_up"], gate_up, n, 2 * I, H)
                g.silu_mul(gate_up, act, n, I)
                g.gemm(act, l["down"], hidden, n, H, I)
        if head:
            g.add_rms_norm_gather(hidden, now, final, b.last, gathered, b.count, H, n, EPS)
            g.gemm(gathered, table, logits, b.count, V, H)

    outputs = {"hidden": _view(hidden, (n, H)), "residual": _view(out_residual, (n, H)),
               "k": _view(kc, (layers, b.blocks, BS, KVH, D)), "v": _view(vc, (layers, b.blocks, BS, KVH, D))}
    if head:
        outputs["logits"] = _view(logits, (b.count, V))
    return {"steps": steps, "outputs": outputs, "keep": (b, w)}


def _prepare_attn_decode(case, x):
    g, b, layers = gpu(), _Batch(case, x).upload(), case["layers"]
    n = b.rows
    kc, vc = _put(x.normal(layers, b.blocks, BS, KVH, D)), _put(x.normal(layers, b.blocks, BS, KVH, D))
    qkv = _put(x.normal(layers, n, HEADS, D))
    qw, kw = _put(x.normal(layers, D, std=0.1, mean=1.0)), _put(x.normal(layers, D, std=0.1, mean=1.0))
    out, rope = _empty((layers, n, QH, D)), _rope_table()
    part = lambda buffer, i: buffer.slice(i * (buffer.bytes // layers), buffer.bytes // layers)  # noqa: E731
    calls = [[part(t, i) for t in (qkv, qw, kw, kc, vc, out)] for i in range(layers)]

    def steps():
        for q, w1, w2, k, v, o in calls:
            g.attention_qkv_rope(q, w1, w2, b.positions, b.slots, k, v, b.ids, b.tables, o, n, QH, KVH, D, BS,
                                 b.blocks, b.stride, b.count, MAX_CTX, EPS, rope, MAX_CTX)

    shape = (layers, b.blocks, BS, KVH, D)
    return {"steps": steps, "keep": (b, qw, kw, qkv),
            "outputs": {"out": _view(out, (layers, n, QH, D)), "k": _view(kc, shape), "v": _view(vc, shape)}}


def _prepare_attn_prefill(case, x):
    g, b = gpu(), _Batch(case, x).upload()
    kc, vc = _put(x.normal(b.blocks, BS, KVH, D)), _put(x.normal(b.blocks, BS, KVH, D))
    q, out = _put(x.normal(b.rows, QH, D)), _empty((b.rows, QH, D))

    def steps():
        g.paged_attention(q, kc, vc, b.positions, b.ids, b.tables, out, b.rows, QH, KVH, D, BS, b.blocks, b.stride,
                          b.count, MAX_CTX)

    return {"steps": steps, "keep": b, "outputs": {"out": _view(out, (b.rows, QH, D))}}


def _prepare_stream(case, x):
    g, n = gpu(), case["tokens"]
    blocks = -(-n // BS)
    order = list(range(blocks))
    x.r.shuffle(order)
    t = torch.arange(n, device="cuda", dtype=torch.int32)
    slots = _put(_i32(order)[(t // BS).long()] * BS + t % BS)
    positions = _put(t % MAX_CTX)
    table = _put(x.normal(32768, H))
    tokens = _put(x.ints(0, 32768, n))
    mlp, attn = _put(x.normal(n, H)), _put(x.normal(n, H))
    qkv, gate_up = _put(x.normal(n, HEADS, D)), _put(x.normal(n, 2, I))
    norm1, norm2 = _put(x.normal(H, std=0.1, mean=1.0)), _put(x.normal(H, std=0.1, mean=1.0))
    qw, kw = _put(x.normal(D, std=0.1, mean=1.0)), _put(x.normal(D, std=0.1, mean=1.0))
    residual, normed1, normed2, query, act = (_empty(s) for s in ((n, H), (n, H), (n, H), (n, QH, D), (n, I)))
    kc, vc, rope = _empty((blocks, BS, KVH, D)), _empty((blocks, BS, KVH, D)), _rope_table()

    def steps():
        g.embedding(tokens, table, residual, n, H, 32768)
        g.add_rms_norm(mlp, residual, norm1, normed1, n, H, EPS)
        g.qkv_rope_cached(qkv, qw, kw, positions, slots, query, kc, vc, n, QH, KVH, D, BS, blocks, EPS, rope, MAX_CTX)
        g.add_rms_norm(attn, residual, norm2, normed2, n, H, EPS)
        g.silu_mul(gate_up, act, n, I)

    shape = (blocks, BS, KVH, D)
    return {"steps": steps, "keep": (slots, order),
            "outputs": {"residual": _view(residual, (n, H)), "normed1": _view(normed1, (n, H)),
                        "normed2": _view(normed2, (n, H)), "query": _view(query, (n, QH, D)), "k": _view(kc, shape),
                        "v": _view(vc, shape), "act": _view(act, (n, I))}}


def _prepare_head(case, x):
    g, n, samples = gpu(), case["rows"], case["samples"]
    hidden, residual, norm = _put(x.normal(n, H)), _put(x.normal(n, H)), _put(x.normal(H, std=0.1, mean=1.0))
    table, rows = _put(x.weight(V, H)), _put(x.ints(0, n, samples))
    gathered, logits = _empty((samples, H)), _empty((samples, V))

    def steps():
        g.add_rms_norm_gather(hidden, residual, norm, rows, gathered, samples, H, n, EPS)
        g.gemm(gathered, table, logits, samples, V, H)

    return {"steps": steps, "outputs": {"gathered": _view(gathered, (samples, H)), "logits": _view(logits, (samples, V))}}


def _prepare_sample(case, x):
    g, n = gpu(), case["rows"]
    logits = _put(x.normal(n, V, std=2.0))
    temps = _put(torch.tensor([0.0 if r < n // 2 else 0.6 for r in range(n)], device="cuda"))
    seeds = [nvr.sampling_seed(x.seed, r, r % 32) for r in range(n)]
    seeds = _put(torch.tensor([s - (1 << 64) if s >> 63 else s for s in seeds], dtype=torch.int64, device="cuda"))
    parts = -(-V // 2048)
    out, scores, ids = _empty((n,), torch.int32), _empty((n, parts), torch.float32), _empty((n, parts), torch.int32)

    def steps():
        g.sample_parallel(logits, temps, seeds, out, scores, ids, n, V)

    return {"steps": steps, "outputs": {"tokens": _view(out, (n,), torch.int32)}}


_PREPARE = {"decode": _prepare_model, "prefill": _prepare_model, "attn_decode": _prepare_attn_decode,
            "attn_prefill": _prepare_attn_prefill, "stream": _prepare_stream, "head": _prepare_head,
            "sample": _prepare_sample}


# --------------------------------------------------------------------- run --
def run(state):
    if "graph" in state:
        state["graph"].replay()
    else:
        state["steps"]()
    return state["outputs"]


# -------------------------------------------------------------------- work --
def work(case):
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": 2 * case["rows"] * V, "flops": case["rows"] * V}
    if kind == "head":
        s = case["samples"]
        return {"bytes": 2 * (V * H + s * V + 3 * s * H), "flops": 2 * s * V * H}
    if kind == "stream":
        # Inputs once, outputs once: table rows, the two branch outputs, qkv, gate_up; residual, two norms, q, k, v, act.
        n = case["tokens"]
        return {"bytes": 2 * n * (3 * H + HEADS * D + 2 * I) + 2 * n * (3 * H + HEADS * D + I), "flops": 60 * n * H}
    seqs = _sequences(case)
    rows, spans = sum(n for _, n in seqs), sum(f + n for f, n in seqs)
    keys = sum(n * f + n * (n + 1) // 2 for f, n in seqs)
    layers = case.get("layers", 1)
    attn = {"bytes": 2 * (2 * spans * KVH * D + 2 * rows * QH * D), "flops": 4 * keys * QH * D}
    if kind == "attn_prefill":
        return attn
    if kind == "attn_decode":
        return {"bytes": layers * (attn["bytes"] + 2 * rows * 4 * KVH * D), "flops": layers * attn["flops"]}
    weights = HEADS * D * H + QH * D * H + 3 * I * H
    total = {"bytes": layers * (2 * weights + 2 * 2 * spans * KVH * D) + 2 * 2 * rows * H,
             "flops": layers * (2 * rows * weights + attn["flops"])}
    if case.get("head"):
        total["bytes"] += 2 * (V * H + len(seqs) * V)
        total["flops"] += 2 * len(seqs) * V * H
    return total


# --------------------------------------------------------------- tolerance --
def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind in ("attn_prefill", "attn_decode", "stream", "head"):
        return {"rel": 4e-3, "max": 0.02}  # one rounding to bf16 of sums in 32 bits
    # Whole layers: four bf16 roundings on the way, and each layer's differences travel through the next.
    return {"rel": 1e-2 if case["layers"] <= 4 else 2.5e-2, "max": 0.2}


# ------------------------------------------------------------------- exact --
def _rms64(x, weight):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * weight.double()


def _rope64(x, positions):
    """x [rows, heads, D] rotated by its row's position."""
    inv = torch.exp(-torch.arange(D // 2, device="cuda", dtype=torch.float64) * (2.0 / D) * math.log(THETA))
    angle = (positions.double()[:, None] * inv)[:, None, :]
    c, s = torch.cos(angle), torch.sin(angle)
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attention64(q, kc, vc, b):
    """q [rows, QH, D] over caches [blocks * BS, KVH, D]."""
    out, at = torch.empty_like(q), 0
    for s, (first, rows) in enumerate(b.seqs):
        ctx = first + rows
        t = torch.arange(ctx, device="cuda")
        place = _i32(b.tables_list[s])[t // BS].long() * BS + t % BS
        k, v = kc[place], vc[place]
        late = t[None, :] > (first + torch.arange(rows, device="cuda"))[:, None]
        for h in range(QH):
            sc = q[at:at + rows, h] @ k[:, h // (QH // KVH)].T.contiguous() / math.sqrt(D)
            p = torch.softmax(sc.masked_fill(late, -math.inf), -1)
            out[at:at + rows, h] = p @ v[:, h // (QH // KVH)].contiguous()
        at += rows
    return out


def _qkv64(qkv, qw, kw, b):
    positions = _i32(b.pos_list)
    q = _rope64(_rms64(qkv[:, :QH], qw), positions)
    k = _rope64(_rms64(qkv[:, QH:QH + KVH], kw), positions)
    return q, k, qkv[:, QH + KVH:]


def _exact_model(case, x):
    b, layers, head = _Batch(case, x), case["layers"], case.get("head", False)
    table_rows = V if head else 4096
    table = x.normal(table_rows, H)
    tokens = x.ints(0, table_rows, b.rows)
    kc, vc = x.normal(layers, b.blocks, BS, KVH, D), x.normal(layers, b.blocks, BS, KVH, D)
    slots, ks, vs = _i32(b.slot_list).long(), [], []
    residual, hidden = table[tokens.long()].double(), None
    for i in range(layers):
        l = _layer_values(x)
        if i:
            residual = residual + hidden
        normed = _rms64(residual, l["input_norm"])
        q, k, v = _qkv64((normed @ l["qkv"].double().T).view(b.rows, HEADS, D), l["q_norm"], l["k_norm"], b)
        k64, v64 = kc[i].double().view(-1, KVH, D), vc[i].double().view(-1, KVH, D)
        k64[slots], v64[slots] = k, v
        attn = _attention64(q, k64, v64, b).view(b.rows, QH * D)
        residual = residual + attn @ l["o_proj"].double().T
        normed = _rms64(residual, l["post_norm"])
        gate, up = (normed @ l["gate_up"].double().T).split(I, -1)
        hidden = (gate * torch.sigmoid(gate) * up) @ l["down"].double().T
        ks.append(k64.view(b.blocks, BS, KVH, D))
        vs.append(v64.view(b.blocks, BS, KVH, D))
    outputs = {"hidden": hidden, "residual": residual, "k": torch.stack(ks), "v": torch.stack(vs)}
    if head:
        last = _rms64(residual + hidden, x.normal(H, std=0.1, mean=1.0))[_i32(b.last_list).long()]
        outputs["logits"] = torch.cat([last @ part.double().T for part in table.split(16384)], -1)
    return outputs


def _exact_attn_decode(case, x):
    b, layers = _Batch(case, x), case["layers"]
    kc, vc = x.normal(layers, b.blocks, BS, KVH, D), x.normal(layers, b.blocks, BS, KVH, D)
    qkv = x.normal(layers, b.rows, HEADS, D)
    qw, kw = x.normal(layers, D, std=0.1, mean=1.0), x.normal(layers, D, std=0.1, mean=1.0)
    slots, out, ks, vs = _i32(b.slot_list).long(), [], [], []
    for i in range(layers):
        q, k, v = _qkv64(qkv[i].double(), qw[i], kw[i], b)
        k64, v64 = kc[i].double().view(-1, KVH, D), vc[i].double().view(-1, KVH, D)
        k64[slots], v64[slots] = k, v
        out.append(_attention64(q, k64, v64, b))
        ks.append(k64.view(b.blocks, BS, KVH, D))
        vs.append(v64.view(b.blocks, BS, KVH, D))
    return {"out": torch.stack(out), "k": torch.stack(ks), "v": torch.stack(vs)}


def _exact_attn_prefill(case, x):
    b = _Batch(case, x)
    kc, vc = x.normal(b.blocks, BS, KVH, D), x.normal(b.blocks, BS, KVH, D)
    q = x.normal(b.rows, QH, D)
    return {"out": _attention64(q.double(), kc.double().view(-1, KVH, D), vc.double().view(-1, KVH, D), b)}


def _exact_stream(case, x):
    n = case["tokens"]
    blocks = -(-n // BS)
    order = list(range(blocks))
    x.r.shuffle(order)
    t = torch.arange(n, device="cuda", dtype=torch.int32)
    slots = (_i32(order)[(t // BS).long()] * BS + t % BS).long()
    table = x.normal(32768, H)
    tokens = x.ints(0, 32768, n)
    mlp, attn = x.normal(n, H).double(), x.normal(n, H).double()
    qkv, gate_up = x.normal(n, HEADS, D).double(), x.normal(n, 2, I).double()
    norm1, norm2 = x.normal(H, std=0.1, mean=1.0), x.normal(H, std=0.1, mean=1.0)
    qw, kw = x.normal(D, std=0.1, mean=1.0), x.normal(D, std=0.1, mean=1.0)
    first = table[tokens.long()].double() + mlp
    second = first + attn
    kc, vc = (torch.zeros(blocks * BS, KVH, D, device="cuda", dtype=torch.float64) for _ in range(2))
    kc[slots] = _rope64(_rms64(qkv[:, QH:QH + KVH], kw), t % MAX_CTX)
    vc[slots] = qkv[:, QH + KVH:]
    gate = gate_up[:, 0]
    return {"residual": second, "normed1": _rms64(first, norm1), "normed2": _rms64(second, norm2),
            "query": _rope64(_rms64(qkv[:, :QH], qw), t % MAX_CTX), "k": kc.view(blocks, BS, KVH, D),
            "v": vc.view(blocks, BS, KVH, D), "act": gate * torch.sigmoid(gate) * gate_up[:, 1]}


def _exact_head(case, x):
    n = case["rows"]
    hidden, residual, norm = x.normal(n, H), x.normal(n, H), x.normal(H, std=0.1, mean=1.0)
    table, rows = x.weight(V, H), x.ints(0, n, case["samples"])
    gathered = _rms64((hidden.double() + residual.double())[rows.long()], norm)
    return {"gathered": gathered, "logits": torch.cat([gathered @ part.double().T for part in table.split(16384)], -1)}


def exact(case, seed):
    """run()'s outputs in 64 bits, without the library; None for token ids, which are no computed numbers."""
    make = {"decode": _exact_model, "prefill": _exact_model, "attn_decode": _exact_attn_decode,
            "attn_prefill": _exact_attn_prefill, "stream": _exact_stream, "head": _exact_head}.get(case["kind"])
    if make is None:
        return None
    outputs = make(dict(case), _Inputs(seed))
    torch.cuda.synchronize()
    return outputs
