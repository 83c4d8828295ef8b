"""The work a user of this package has it do, as cases that can be timed and
checked: the packed projections, the MoE block, the attention layers of a
prompt's chunk, the output head, the sampler, and whole decode steps and
prefills of a four-layer hybrid stack (three Gated DeltaNet layers, one full
attention layer, each with the 256-expert MoE block).

Geometry is the checkpoint's (hidden 2048, experts of 512, top 8 of 256);
weights are packed codes drawn uniformly with lognormal scales, as the codecs
store them, and inputs are RMS-normalised rows. Sizes run over what the
entry points serve: 1 to 32 sequences a decode step, chunks of 1 to 2048
tokens, histories up to 4096 positions.
"""
import math

import numpy as np
import torch

from adi_amd import hip

DEVICE = "cuda:0"
HIDDEN, EXPERT_HIDDEN, EXPERTS, TOP = 2048, 512, 256, 8
QUERY_HEADS, KV_HEADS, HEAD = 16, 2, 256
KEY_HEADS, VALUE_HEADS, LINEAR_HEAD = 16, 32, 128
CHANNELS = 8192
VOCAB = 151936          # the output head of the package's benchmark
SAMPLER_VOCAB = 248320  # the checkpoint's vocabulary
LAYERS = 4              # three Gated DeltaNet layers, then one full attention

NE_SHAPES = ((512, 2048), (2048, 512), (2048, 2048), (4096, 2048), (8192, 2048), (2048, 4096))


# ---- the cases -----------------------------------------------------------------

def listed():
    return [
        # the smallest call: one shared-expert projection of a decode token,
        # where the launch itself counts
        {"name": "projection_1", "kind": "projection", "rows": 512, "columns": 2048, "batch": 1},
        # the MoE block of one sequence's decode step
        {"name": "moe_1", "kind": "moe", "tokens": 1, "zipf": False},
        # the MoE block of a serving step over many sequences (a ragged count)
        {"name": "moe_45", "kind": "moe", "tokens": 45, "zipf": False},
        # the MoE block of a large prefill micro-batch with skewed routing
        {"name": "moe_512", "kind": "moe", "tokens": 512, "zipf": True},
        # full attention over a late chunk of a 4096-token prompt
        {"name": "full_attention_512", "kind": "full", "position": 3584, "count": 512},
        # Gated DeltaNet over a chunk of a prompt
        {"name": "linear_attention_512", "kind": "linear", "count": 512},
        # the int5 output head for one sequence and for a serving step
        {"name": "head_1", "kind": "head", "batch": 1},
        {"name": "head_16", "kind": "head", "batch": 16},
        # top-p sampling of a serving step's logits
        {"name": "top_p_16", "kind": "sample", "rows": 16, "temperature": 0.7, "top_p": 0.9},
        # whole calls: a decode step of one sequence (interactive use), a
        # decode step of 32 sequences at mixed positions (serving), and a
        # prompt at the default micro-batch
        {"name": "decode_1", "kind": "decode", "batch": 1, "context": 2000},
        {"name": "decode_32", "kind": "decode", "batch": 32, "context": 2000},
        {"name": "prefill_1500", "kind": "prefill", "tokens": 1500, "ubatch": 0},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("projection", "moe", "moe", "full", "full", "linear", "head", "sample",
                       "decode", "decode", "prefill"))
    if kind == "projection":
        rows, columns = rng.choice(NE_SHAPES)
        return {"kind": kind, "rows": rows, "columns": columns, "batch": _log(rng, 1, 512)}
    if kind == "moe":
        tokens = _log(rng, 1, 2048)
        return {"kind": kind, "tokens": tokens, "zipf": tokens >= 64 and rng.random() < 0.5}
    if kind == "full":
        count = _log(rng, 1, 1024)
        # no more work than the listed chunk
        last = min(4096, 512 * 4096 // count)
        return {"kind": kind, "position": max(0, _log(rng, max(count, 16), last) - count), "count": count}
    if kind == "linear":
        return {"kind": kind, "count": _log(rng, 1, 1024)}
    if kind == "head":
        return {"kind": kind, "batch": _log(rng, 1, 32)}
    if kind == "sample":
        return {"kind": kind, "rows": _log(rng, 1, 32), "temperature": rng.choice((0.0, 0.6, 0.7, 1.0)),
                "top_p": rng.choice((0.8, 0.9, 0.95))}
    if kind == "decode":
        return {"kind": kind, "batch": _log(rng, 1, 32), "context": _log(rng, 64, 4096)}
    return {"kind": kind, "tokens": _log(rng, 16, 1500), "ubatch": rng.choice((0, 0, 256, 512))}


# ---- inputs: plain device tensors from the seed ----------------------------------

class _Draw:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(seed)

    def words(self, n):
        return torch.randint(-32768, 32768, (n,), dtype=torch.int16, device=DEVICE, generator=self.g)

    def normal(self, shape, scale=1.0, loc=0.0):
        return torch.randn(shape, device=DEVICE, generator=self.g) * scale + loc

    def scales(self, n):
        return self.normal((n,), 0.5).exp().half()

    def bf16(self, shape, scale, loc=0.0):
        return self.normal(shape, scale, loc).to(torch.bfloat16)

    def signs(self, n):
        return (torch.randint(0, 2, (n,), device=DEVICE, generator=self.g) * 2 - 1).to(torch.int8)

    def uniform(self, n):
        return torch.rand(n, device=DEVICE, generator=self.g) * 2 - 1

    def scalar(self):
        return float(np.float32(math.exp(0.5 * float(self.normal((1,))))))

    def rows(self, count, n=HIDDEN):
        x = self.normal((count, n))
        return x / x.square().mean(1, keepdim=True).add(1e-6).sqrt()


def _ne(d, rows, columns):
    tiles = (rows // 16) * (columns // 16)
    return {"rows": rows, "columns": columns, "trellis": d.words(tiles * 64), "su": d.signs(columns),
            "sv": d.signs(rows), "scale": d.scalar()}


def _experts(d, rows, columns):
    tiles = (rows // 16) * (columns // 16)
    return {"rows": rows, "columns": columns, "trellis": d.words(EXPERTS * tiles * 24),
            "su": d.scales(EXPERTS * columns), "sv": d.scales(EXPERTS * rows),
            "gamma": d.scales(EXPERTS * (rows // 16 + columns // 16))}


def _tluts(d):
    return {"expert": d.uniform(32768 * 8), "ne": d.uniform(512 * 2)}


def _moe(d):
    return {"router": d.bf16((EXPERTS, HIDDEN), 0.02), "shared_expert_gate": d.bf16((1, HIDDEN), 0.02),
            "gate": _experts(d, EXPERT_HIDDEN, HIDDEN), "up": _experts(d, EXPERT_HIDDEN, HIDDEN),
            "down": _experts(d, HIDDEN, EXPERT_HIDDEN), "shared_gate": _ne(d, EXPERT_HIDDEN, HIDDEN),
            "shared_up": _ne(d, EXPERT_HIDDEN, HIDDEN), "shared_down": _ne(d, HIDDEN, EXPERT_HIDDEN)}


def _full(d):
    return {"query": _ne(d, QUERY_HEADS * 2 * HEAD, HIDDEN), "key": _ne(d, KV_HEADS * HEAD, HIDDEN),
            "value": _ne(d, KV_HEADS * HEAD, HIDDEN), "output": _ne(d, HIDDEN, QUERY_HEADS * HEAD),
            "query_norm": d.bf16((HEAD,), 0.2), "key_norm": d.bf16((HEAD,), 0.2)}


def _linear(d):
    alpha_bias = d.bf16((VALUE_HEADS,), 1.0)
    alpha_bias[:2] = torch.tensor([22.0, 25.0])  # both branches of the softplus
    return {"qkv": _ne(d, CHANNELS, HIDDEN), "gate": _ne(d, VALUE_HEADS * LINEAR_HEAD, HIDDEN),
            "output": _ne(d, HIDDEN, VALUE_HEADS * LINEAR_HEAD), "alpha": d.bf16((VALUE_HEADS, HIDDEN), 0.02),
            "beta": d.bf16((VALUE_HEADS, HIDDEN), 0.02), "convolution": d.bf16((CHANNELS, 4), 0.5),
            "alpha_bias": alpha_bias, "a_log": d.bf16((VALUE_HEADS,), 0.5, -1.0),
            "norm": d.bf16((LINEAR_HEAD,), 0.1, 1.0)}


def _head(d):
    packed = torch.randint(0, 256, (VOCAB * HIDDEN // 8 * 5,), dtype=torch.uint8, device=DEVICE, generator=d.g)
    return {"packed": packed, "scales": d.scales(VOCAB * HIDDEN // 64)}


def _model(d):
    groups = VOCAB * HIDDEN // 64
    minimum = d.normal((groups,), 0.02, -0.06).half()
    return {"tluts": _tluts(d),
            "layers": [{"input_norm": d.bf16((HIDDEN,), 0.1), "post_norm": d.bf16((HIDDEN,), 0.1),
                        "attention": _full(d) if i == LAYERS - 1 else _linear(d), "moe": _moe(d)}
                       for i in range(LAYERS)],
            "embedding": {"packed": torch.randint(0, 256, (VOCAB * HIDDEN // 2,), dtype=torch.uint8,
                                                  device=DEVICE, generator=d.g),
                          "minimum": minimum,
                          "maximum": (minimum.float() + d.normal((groups,), 0.03, 0.1).abs()).half()},
            "final_norm": d.bf16((HIDDEN,), 0.1), "head": _head(d)}


def _tokens(d, count):
    return [int(t) for t in torch.randint(0, VOCAB, (count,), device=DEVICE, generator=d.g).tolist()]


def _positions(case):
    """A serving batch's positions: spread from a quarter of the context to all of it."""
    n, c = case["batch"], case["context"]
    return [c - 1 - (3 * c // 4) * b // n for b in range(n)]


def _inputs(case, seed):
    d, kind = _Draw(seed), case["kind"]
    if kind == "projection":
        return {"tluts": _tluts(d), "matrix": _ne(d, case["rows"], case["columns"]),
                "x": d.rows(case["batch"], case["columns"])}
    if kind == "moe":
        bias = None
        if case["zipf"]:  # the routing skew of the benchmark's prefill workloads
            rank = torch.randperm(EXPERTS, device=DEVICE, generator=d.g) + 1
            bias = -1.1 * torch.log(rank.float())
        return {"tluts": _tluts(d), "moe": _moe(d), "bias": bias, "x": d.rows(case["tokens"])}
    if kind == "full":
        shape = (case["position"] + case["count"], KV_HEADS, HEAD)
        return {"tluts": _tluts(d), "attention": _full(d), "x": d.rows(case["count"]),
                "keys": d.normal(shape), "values": d.normal(shape)}
    if kind == "linear":
        return {"tluts": _tluts(d), "attention": _linear(d), "x": d.rows(case["count"]),
                "conv": d.normal((CHANNELS, 3)), "rec": d.normal((VALUE_HEADS, LINEAR_HEAD, LINEAR_HEAD), 0.05)}
    if kind == "head":
        return {"head": _head(d), "x": d.rows(case["batch"])}
    if kind == "sample":
        logits = d.normal((case["rows"], SAMPLER_VOCAB), 2.0)
        likely = torch.randint(0, SAMPLER_VOCAB, (16,), device=DEVICE, generator=d.g)
        logits[:, likely] += 12.0  # a few likely tokens over a normal tail
        words = torch.randint(0, 1 << 62, (case["rows"],), device=DEVICE, generator=d.g)
        return {"logits": logits, "words": words}
    if kind == "decode":
        n, c = case["batch"], case["context"]
        # sequence b's cache starts c - 1 - position rows into its part, so
        # every new entry is the part's last row
        return {"model": _model(d), "tokens": _tokens(d, n), "keys": d.normal((n, c, KV_HEADS, HEAD)),
                "values": d.normal((n, c, KV_HEADS, HEAD)), "conv": d.normal((LAYERS - 1, n, CHANNELS, 3)),
                "rec": d.normal((LAYERS - 1, n, VALUE_HEADS, LINEAR_HEAD, LINEAR_HEAD), 0.05)}
    return {"model": _model(d), "tokens": _tokens(d, case["tokens"])}


# ---- the package's descriptors over them ------------------------------------------

_CONTEXT = []


def _context():
    """One context for the program, as a server keeps it."""
    if not _CONTEXT:
        _CONTEXT.append(hip.Context(0))
    return _CONTEXT[0]


def _book(ctx, tluts, kind):
    make = ctx.expert_codebook if kind == "expert" else ctx.ne_codebook
    return make(tluts[kind].cpu().numpy())


def _ne_struct(m, book):
    return hip.NeMatrix(m["rows"], m["columns"], m["trellis"].data_ptr(), m["su"].data_ptr(),
                        m["sv"].data_ptr(), m["scale"], book)


def _bf16_struct(t):
    return hip.Bf16Matrix(t.shape[0], t.shape[1], t.data_ptr())


def _stack_struct(m):
    return hip.ExpertStack(m["trellis"].data_ptr(), m["su"].data_ptr(), m["sv"].data_ptr(), m["gamma"].data_ptr())


def _moe_struct(m, books):
    return hip.MoeLayer(HIDDEN, EXPERT_HIDDEN, EXPERTS, _bf16_struct(m["router"]),
                        _bf16_struct(m["shared_expert_gate"]), _stack_struct(m["gate"]), _stack_struct(m["up"]),
                        _stack_struct(m["down"]), books[0], *(_ne_struct(m[k], books[1]) for k in
                                                              ("shared_gate", "shared_up", "shared_down")))


def _full_struct(m, book):
    return hip.FullAttentionStruct(*(_ne_struct(m[k], book) for k in ("query", "key", "value", "output")),
                                   m["query_norm"].data_ptr(), m["key_norm"].data_ptr())


def _linear_struct(m, book):
    return hip.LinearAttentionStruct(*(_ne_struct(m[k], book) for k in ("qkv", "gate", "output")),
                                     _bf16_struct(m["alpha"]), _bf16_struct(m["beta"]),
                                     *(m[k].data_ptr() for k in ("convolution", "alpha_bias", "a_log", "norm")))


def _head_struct(h):
    return hip.HeadChunk(VOCAB, HIDDEN, h["packed"].data_ptr(), h["scales"].data_ptr(), None, None, 0)


def _model_of(ctx, m):
    books = (_book(ctx, m["tluts"], "expert"), _book(ctx, m["tluts"], "ne"))
    layers = []
    for i, L in enumerate(m["layers"]):
        full = i == LAYERS - 1
        layers.append(hip.DeviceDecoderLayer(hip.DecoderLayerStruct(
            L["input_norm"].data_ptr(), L["post_norm"].data_ptr(), int(full),
            _full_struct(L["attention"], books[1]) if full else hip.FullAttentionStruct(),
            hip.LinearAttentionStruct() if full else _linear_struct(L["attention"], books[1]),
            _moe_struct(L["moe"], books)), ()))
    e = m["embedding"]
    embedding = hip.DeviceEmbedding(hip.Embedding(VOCAB, HIDDEN, e["packed"].data_ptr(), e["minimum"].data_ptr(),
                                                  e["maximum"].data_ptr(), None, None, 0), ())
    return hip.Model(layers, embedding, m["final_norm"], [hip.DeviceHead(_head_struct(m["head"]), ())])


class _Sequence:
    """A sequence over state tensors the program owns: keys and values at the
    given addresses, one convolution and recurrent state per linear layer."""

    def __init__(self, position, keys, values, capacity, conv, rec):
        self._layers = (hip.LayerState * LAYERS)()
        for i in range(LAYERS - 1):
            self._layers[i] = hip.LayerState(None, None, 0, conv[i].data_ptr(), rec[i].data_ptr())
        self._layers[LAYERS - 1] = hip.LayerState(keys, values, capacity, None, None)
        self.start = position
        self.struct = hip.DecoderStateStruct(position, self._layers)


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    s = _inputs(case, seed)
    s.update(case=case, ctx=ctx)

    def new(*shape, dtype=torch.float32):
        return torch.empty(shape, dtype=dtype, device=DEVICE)

    if kind == "projection":
        s["device"] = hip.DeviceNe(_ne_struct(s["matrix"], _book(ctx, s["tluts"], "ne")), ())
        s["out"] = new(case["batch"], case["rows"])
    elif kind == "moe":
        books = (_book(ctx, s["tluts"], "expert"), _book(ctx, s["tluts"], "ne"))
        s["device"] = hip.DeviceMoeLayer(_moe_struct(s["moe"], books), (), EXPERTS, HIDDEN)
        s["out"] = new(case["tokens"], HIDDEN)
        s["experts"] = new(case["tokens"], TOP, dtype=torch.int32)
        s["weights"] = new(case["tokens"], TOP)
    elif kind == "full":
        s["device"] = hip.DeviceFullAttention(_full_struct(s["attention"], _book(ctx, s["tluts"], "ne")), ())
        s["out"] = new(case["count"], HIDDEN)
    elif kind == "linear":
        s["device"] = hip.DeviceLinearAttention(_linear_struct(s["attention"], _book(ctx, s["tluts"], "ne")), ())
        s["out"] = new(case["count"], HIDDEN)
    elif kind == "head":
        s["device"] = hip.DeviceHead(_head_struct(s["head"]), ())
        s["out"] = new(case["batch"], VOCAB)
    elif kind == "sample":
        s["out"] = new(case["rows"], dtype=torch.int32)
    elif kind == "decode":
        s["device"] = _model_of(ctx, s["model"])
        entry = KV_HEADS * HEAD * 4
        s["sequences"] = []
        for b, p in enumerate(_positions(case)):
            skip = (b * case["context"] + case["context"] - 1 - p) * entry
            s["sequences"].append(_Sequence(p, s["keys"].data_ptr() + skip, s["values"].data_ptr() + skip, p + 1,
                                            s["conv"][:, b], s["rec"][:, b]))
        s["out"] = new(case["batch"], VOCAB)
    else:
        s["device"] = _model_of(ctx, s["model"])
        n = case["tokens"]
        s["keys"], s["values"] = new(n, KV_HEADS, HEAD), new(n, KV_HEADS, HEAD)
        s["conv"], s["rec"] = new(LAYERS - 1, CHANNELS, 3), new(LAYERS - 1, VALUE_HEADS, LINEAR_HEAD, LINEAR_HEAD)
        s["sequence"] = _Sequence(0, s["keys"].data_ptr(), s["values"].data_ptr(), n, s["conv"], s["rec"])
        s["out"] = new(VOCAB)
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "projection":
        hip.ne_matmul(ctx, s["device"], s["x"], case["batch"], s["out"])
        return s["out"]
    if kind == "moe":
        hip.moe_forward(ctx, s["device"], s["x"], case["tokens"], s["bias"], s["out"], s["experts"], s["weights"])
        return {"out": s["out"], "experts": s["experts"], "weights": s["weights"]}
    if kind == "full":
        p, n = case["position"], case["count"]
        hip.full_attention_prefill(ctx, s["device"], p, n, s["x"], s["out"], s["keys"], s["values"], p + n)
        return {"out": s["out"], "keys": s["keys"][p:], "values": s["values"][p:]}
    if kind == "linear":
        hip.linear_attention_prefill(ctx, s["device"], case["count"], s["x"], s["out"], s["conv"], s["rec"])
        return {"out": s["out"], "conv": s["conv"], "rec": s["rec"]}
    if kind == "head":
        hip.head_matmul(ctx, s["device"], s["x"], case["batch"], s["out"])
        return s["out"]
    if kind == "sample":
        hip.sample_rows(ctx, s["logits"], case["rows"], SAMPLER_VOCAB, case["temperature"], case["top_p"],
                        s["words"], s["out"])
        return s["out"]
    if kind == "decode":
        for q in s["sequences"]:  # the same step again
            q.struct.position = q.start
        hip.decode_batch(ctx, s["device"], s["tokens"], s["sequences"], s["out"])
        return {"logits": s["out"], "keys": s["keys"][:, -1], "values": s["values"][:, -1],
                "conv": s["conv"], "rec": s["rec"]}
    s["sequence"].struct.position = 0  # a new prompt: its linear states start at zero
    s["conv"].zero_()
    s["rec"].zero_()
    hip.prefill(ctx, s["device"], s["tokens"], s["sequence"], s["out"], case["ubatch"])
    return {"logits": s["out"], "keys": s["keys"], "values": s["values"], "conv": s["conv"], "rec": s["rec"]}


# ---- what a pass cannot do without ------------------------------------------------

def _ne_work(rows, columns, batch):
    return rows * columns // 2 + rows + columns, 2 * rows * columns * batch


def _active(tokens, zipf):
    """Experts that `tokens` rows route to, for normal logits of the router's spread."""
    rng = np.random.default_rng(7)
    bias = -1.1 * np.log(np.arange(EXPERTS) + 1.0) if zipf else 0.0
    logits = rng.normal(0.0, 0.02 * math.sqrt(HIDDEN), (tokens, EXPERTS)) + bias
    return len(np.unique(np.argpartition(-logits, TOP, axis=1)[:, :TOP]))


def _moe_work(tokens, zipf=False):
    expert = 3 * (EXPERT_HIDDEN * HIDDEN * 3 // 16 + 2 * (EXPERT_HIDDEN + HIDDEN) + 2 * (EXPERT_HIDDEN + HIDDEN) // 16)
    shared = [_ne_work(*shape, tokens) for shape in ((512, 2048), (512, 2048), (2048, 512))]
    nbytes = (EXPERTS + 1) * HIDDEN * 2 + _active(tokens, zipf) * expert + sum(b for b, _ in shared)
    flops = tokens * (TOP * 3 * 2 * EXPERT_HIDDEN * HIDDEN + 2 * (EXPERTS + 1) * HIDDEN) + sum(f for _, f in shared)
    return nbytes, flops


def _full_work(positions):
    """Full attention of one token at each of `positions` (projections of all of them together)."""
    n = len(positions)
    parts = [_ne_work(*shape, n) for shape in ((8192, HIDDEN), (512, HIDDEN), (512, HIDDEN), (HIDDEN, 4096))]
    seen = sum(p + 1 for p in positions)
    return sum(b for b, _ in parts), sum(f for _, f in parts) + 4 * QUERY_HEADS * HEAD * seen


def _linear_work(tokens):
    parts = [_ne_work(*shape, tokens) for shape in ((8192, HIDDEN), (4096, HIDDEN), (HIDDEN, 4096))]
    state = VALUE_HEADS * LINEAR_HEAD * LINEAR_HEAD
    return sum(b for b, _ in parts) + 64 * HIDDEN * 2 + CHANNELS * 8, sum(f for _, f in parts) + 7 * state * tokens


_STATE = 2 * 4 * (VALUE_HEADS * LINEAR_HEAD * LINEAR_HEAD + CHANNELS * 3)  # a linear layer's state, read and written
_ENTRY = 2 * KV_HEADS * HEAD * 4                                           # a position's key and value


def _head_work(batch):
    return VOCAB * HIDDEN * 5 // 8 + VOCAB * HIDDEN // 32 + 4 * batch * (HIDDEN + VOCAB), 2 * VOCAB * HIDDEN * batch


def work(case):
    kind = case["kind"]
    if kind == "projection":
        b, f = _ne_work(case["rows"], case["columns"], case["batch"])
        b += 4 * case["batch"] * (case["rows"] + case["columns"])
    elif kind == "moe":
        b, f = _moe_work(case["tokens"], case["zipf"])
        b += 8 * case["tokens"] * (HIDDEN + TOP)
    elif kind == "full":
        p, n = case["position"], case["count"]
        b, f = _full_work(range(p, p + n))
        b += 8 * n * HIDDEN + _ENTRY * (p + n)
    elif kind == "linear":
        b, f = _linear_work(case["count"])
        b += 8 * case["count"] * HIDDEN + _STATE
    elif kind == "head":
        b, f = _head_work(case["batch"])
    elif kind == "sample":
        b, f = 4 * case["rows"] * SAMPLER_VOCAB, 2 * case["rows"] * SAMPLER_VOCAB
    else:
        if kind == "decode":
            positions, n, sequences = _positions(case), case["batch"], case["batch"]
            cache = sum(p + 1 for p in positions)
        else:
            n, sequences = case["tokens"], 1
            positions, cache = range(n), n
        parts = [_linear_work(n)] * (LAYERS - 1) + [_full_work(positions)] + [_moe_work(n)] * LAYERS
        parts.append(_head_work(sequences))
        b = sum(x for x, _ in parts) + (LAYERS - 1) * sequences * _STATE + _ENTRY * cache + n * HIDDEN // 2
        f = sum(x for _, x in parts)
    return {"bytes": b, "flops": f}


def tolerance(case):
    # about four times the largest difference from exact() seen over the ranges
    kind = case["kind"]
    if kind == "sample":
        return "exact"  # token ids
    if kind in ("projection", "head"):
        return {"rel": 2e-6, "max": 3e-5}  # one 32-bit sum an output
    if kind in ("moe", "full", "linear"):
        return {"rel": 5e-6, "max": 2e-4, "differ": 0.0}  # chains of a few 32-bit sums
    if kind == "decode":
        return {"rel": 2e-5, "max": 2e-3}
    # 1,500 tokens through four layers' routers: a token whose eighth and
    # ninth experts tie to the last bits may take the other one, which moves
    # that token's rows in the layers behind by some percent
    return {"rel": 1e-2, "max": 0.9}


# ---- the same in 64 bits ------------------------------------------------------------

def _hadamard64(v):
    n, lead = v.shape[-1], v.shape[:-1]
    h = 1
    while h < n:
        v = v.reshape(*lead, n // (2 * h), 2, h)
        v = torch.stack((v[..., 0, :] + v[..., 1, :], v[..., 0, :] - v[..., 1, :]), -2)
        h *= 2
    return v.reshape(*lead, n) / math.sqrt(n)


def _states(trellis, words, step):
    """The 16-bit windows of each tile's bit stream, one every `step` bits."""
    w = trellis.long().bitwise_and(0xFFFF).reshape(-1, words)
    at = torch.arange(words * 16 // step, device=DEVICE) * step
    word, offset = at // 16, at % 16
    pair = (w[:, word] << 16) | w[:, (word + 1) % words]
    return (pair >> (16 - offset)) & 0xFFFF


def _values(states, tlut, width):
    product = states * (states + 1)
    row = product & 0x7FFF if width == 8 else (product >> 6) & 0x1FF
    v = tlut.half().double().reshape(-1, width)[row]
    v[..., 0] *= 1.0 - 2.0 * ((product >> 15) & 1)
    return v


def _weights64(v, rows, columns):
    """Tiles of 16 x 16 values, tile rows first, to a matrix."""
    return v.reshape(rows // 16, columns // 16, 16, 16).transpose(1, 2).reshape(rows, columns)


def _ne64(m, tlut, x):
    w = _weights64(_values(_states(m["trellis"], 64, 8), tlut, 2), m["rows"], m["columns"]) * m["scale"]
    return _hadamard64(_hadamard64(x * m["su"].double()) @ w.T) * m["sv"].double()


def _expert64(m, tlut, e, x):
    rows, columns = m["rows"], m["columns"]
    tr, tc = rows // 16, columns // 16
    part = {k: m[k].reshape(EXPERTS, -1)[e] for k in ("trellis", "su", "sv", "gamma")}
    w = _weights64(_values(_states(part["trellis"], 24, 12), tlut, 8), rows, columns)
    diagonal = torch.arange(tr, device=DEVICE)[:, None] + torch.arange(tc, device=DEVICE)[None]
    wave = tr + tc - 1 - diagonal - (diagonal >= tc).long()
    gamma = part["gamma"].double()[wave].repeat_interleave(16, 0).repeat_interleave(16, 1)
    return _hadamard64(_hadamard64(x * part["su"].double()) @ (w * gamma).T) * part["sv"].double()


def _silu(v):
    return v * torch.sigmoid(v)


def _moe64(m, tluts, x, bias=None):
    logits = x @ m["router"].double().T
    if bias is not None:
        logits = logits + bias.double()
    top, chosen = logits.topk(TOP, dim=1)
    weights = torch.softmax(top, 1)
    out = torch.zeros_like(x)
    for e in torch.unique(chosen).tolist():
        token, route = (chosen == e).nonzero(as_tuple=True)
        rows = x[token]
        hidden = _silu(_expert64(m["gate"], tluts["expert"], e, rows)) * _expert64(m["up"], tluts["expert"], e, rows)
        out[token] += weights[token, route, None] * _expert64(m["down"], tluts["expert"], e, hidden)
    hidden = _silu(_ne64(m["shared_gate"], tluts["ne"], x)) * _ne64(m["shared_up"], tluts["ne"], x)
    shared = _ne64(m["shared_down"], tluts["ne"], hidden)
    return out + torch.sigmoid(x @ m["shared_expert_gate"].double().T) * shared, weights


def _norm64(x, weight, offset):
    return x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt() * (offset + weight.double())


def _rope64(v, positions):
    """The model's angles are single-precision quotients; everything after them is in 64 bits."""
    divisor = np.power(np.float64(1e7), np.arange(32) / 32.0).astype(np.float32)
    theta = np.array(positions, np.float32)[:, None] / divisor
    angle = torch.from_numpy(theta.astype(np.float64)).to(DEVICE)[:, None]
    a, b = v[..., :32], v[..., 32:64]
    return torch.cat((a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin(), v[..., 64:]), -1)


def _full64(m, tlut, x, positions, keys, values):
    """x[i] at positions[i] over history keys[i], values[i] ([positions[i]] entries, in 64 bits), or, with
    one history for all, the chunk after it. Returns the outputs and the new entries."""
    n = x.shape[0]
    q = _ne64(m["query"], tlut, x).reshape(n, QUERY_HEADS, 2, HEAD)
    query, gate = _rope64(_norm64(q[:, :, 0], m["query_norm"], 1.0), positions), q[:, :, 1]
    k = _ne64(m["key"], tlut, x).reshape(n, KV_HEADS, HEAD)
    k = _rope64(_norm64(k, m["key_norm"], 1.0), positions)
    v = _ne64(m["value"], tlut, x).reshape(n, KV_HEADS, HEAD)
    attended = torch.empty(n, QUERY_HEADS, HEAD, dtype=torch.float64, device=DEVICE)
    chunk = not isinstance(keys, list)
    for i in range(1 if chunk else n):
        rows = slice(0, n) if chunk else slice(i, i + 1)
        ks = torch.cat(((keys if chunk else keys[i]).double(), k[rows]))
        vs = torch.cat(((values if chunk else values[i]).double(), v[rows]))
        at = torch.tensor(positions[rows], device=DEVICE)[:, None]
        past = torch.arange(ks.shape[0], device=DEVICE)[None] > at
        for h in range(QUERY_HEADS):
            kv = h // (QUERY_HEADS // KV_HEADS)
            score = (query[rows, h] @ ks[:, kv].T / 16.0).masked_fill(past, -math.inf)
            attended[rows, h] = torch.softmax(score, 1) @ vs[:, kv]
    return _ne64(m["output"], tlut, (attended * torch.sigmoid(gate)).reshape(n, -1)), k, v


def _linear64(m, tlut, x, conv, rec, chunk):
    """x[i] of sequence i (conv and rec [n, ...]), or with `chunk` x's rows in order through one state."""
    n = x.shape[0]
    qkv = _ne64(m["qkv"], tlut, x)
    gate = _ne64(m["gate"], tlut, x).reshape(n, VALUE_HEADS, LINEAR_HEAD)
    weight = m["convolution"].double()
    if chunk:
        line = torch.cat((conv[0].T, qkv))  # [3 + n, channels]
        y = sum(line[i:i + n] * weight[:, i] for i in range(4))
        conv = line[n:].T[None]
    else:
        line = torch.cat((conv, qkv[:, :, None]), 2)
        y = (line * weight).sum(2)
        conv = line[:, :, 1:]
    y = _silu(y)
    qk = y[:, :4096].reshape(n, 2, KEY_HEADS, LINEAR_HEAD)
    qk = qk / (qk.square().sum(-1, keepdim=True) + 1e-6).sqrt()
    q, k = qk.repeat_interleave(VALUE_HEADS // KEY_HEADS, 2).unbind(1)
    v = y[:, 4096:].reshape(n, VALUE_HEADS, LINEAR_HEAD)
    beta = torch.sigmoid(x @ m["beta"].double().T)
    rate = torch.nn.functional.softplus(x @ m["alpha"].double().T + m["alpha_bias"].double(), threshold=1e9)
    decay = torch.exp(-m["a_log"].double().exp() * rate)

    def step(state, i):
        state = state * decay[i, :, None, None]
        delta = (v[i] - (state @ k[i, ..., None])[..., 0]) * beta[i, :, None]
        state = state + delta[..., None] * k[i, :, None]
        return state, (state @ q[i, ..., None])[..., 0] / math.sqrt(LINEAR_HEAD)

    out, states, state = [], [], rec[0]
    for i in range(n):
        state, o = step(state if chunk else rec[i], i)
        out.append(o)
        if not chunk:
            states.append(state)
    o = _norm64(torch.stack(out), m["norm"], 0.0) * _silu(gate)
    return _ne64(m["output"], tlut, o.reshape(n, -1)), conv, state[None] if chunk else torch.stack(states)


def _head64(h, x):
    out = []
    for part in range(8):
        rows = VOCAB // 8
        packed = h["packed"].reshape(VOCAB, HIDDEN // 8, 5)[part * rows:(part + 1) * rows].long()
        word = sum(packed[..., i] << (8 * i) for i in range(5))
        codes = torch.stack([(word >> (5 * i)) & 31 for i in range(8)], -1).reshape(rows, HIDDEN // 64, 64) - 16
        scale = h["scales"].reshape(VOCAB, HIDDEN // 64, 1)[part * rows:(part + 1) * rows].double()
        out.append(x @ (codes * scale).reshape(rows, HIDDEN).T)
    return torch.cat(out, 1)


def _embedding64(e, tokens):
    at = torch.tensor(tokens, device=DEVICE)
    packed = e["packed"].reshape(VOCAB, HIDDEN // 2)[at].long()
    codes = torch.stack((packed >> 4, packed & 15), -1).reshape(len(tokens), HIDDEN // 64, 64).double()
    low = e["minimum"].reshape(VOCAB, HIDDEN // 64)[at].double()
    high = e["maximum"].reshape(VOCAB, HIDDEN // 64)[at].double()
    step = (high - low).clamp_min(1e-8) / 15.0
    return (low[..., None] + codes * step[..., None]).reshape(len(tokens), HIDDEN)


def exact(case, seed):
    kind = case["kind"]
    # a token id has no 64-bit value, and a prompt's routes that tie to the
    # last bits (see tolerance) would stand for all of a prefill's difference;
    # its layers are measured by the cases of their own
    if kind in ("sample", "prefill"):
        return None
    s = _inputs(case, seed)
    if kind == "head":
        return _head64(s["head"], s["x"].double())
    if kind == "decode":
        m, positions = s["model"], _positions(case)
        tluts = m["tluts"]
        hidden = _embedding64(m["embedding"], s["tokens"])
        first = [case["context"] - 1 - p for p in positions]
        keys = [s["keys"][b, f:-1] for b, f in enumerate(first)]
        values = [s["values"][b, f:-1] for b, f in enumerate(first)]
        convs, recs = [], []
        for i, L in enumerate(m["layers"]):
            x = _norm64(hidden, L["input_norm"], 1.0)
            if i == LAYERS - 1:
                out, k, v = _full64(L["attention"], tluts["ne"], x, positions, keys, values)
            else:
                out, conv, rec = _linear64(L["attention"], tluts["ne"], x, s["conv"][i].double(),
                                           s["rec"][i].double(), False)
                convs.append(conv)
                recs.append(rec)
            hidden = hidden + out
            hidden = hidden + _moe64(L["moe"], tluts, _norm64(hidden, L["post_norm"], 1.0))[0]
        return {"logits": _head64(m["head"], _norm64(hidden, m["final_norm"], 1.0)), "keys": k, "values": v,
                "conv": torch.stack(convs), "rec": torch.stack(recs)}
    x, tluts = s["x"].double(), s["tluts"]
    if kind == "projection":
        return _ne64(s["matrix"], tluts["ne"], x)
    if kind == "moe":
        out, weights = _moe64(s["moe"], tluts, x, s["bias"])
        return {"out": out, "experts": None, "weights": weights}
    if kind == "full":
        p = case["position"]
        out, k, v = _full64(s["attention"], tluts["ne"], x, list(range(p, p + case["count"])), s["keys"][:p],
                            s["values"][:p])
        return {"out": out, "keys": k, "values": v}
    out, conv, rec = _linear64(s["attention"], tluts["ne"], x, s["conv"].double()[None], s["rec"].double()[None], True)
    return {"out": out, "conv": conv[0], "rec": rec[0]}
