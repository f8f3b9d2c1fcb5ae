"""The calls by which this framework's speed is judged.

A case is one call (or the few calls of one layer, or one step of an engine) of the
paged KV cache and its attention, through `chibillm_amd.ckv`, on inputs a serving
program has in hand: a pool whose pages are scattered, an uploaded batch, and the
layer's new rows. Values are N(0, 1) from the seed, as the benchmark's are.

`listed()` are fixed sizes; `draw(rng)` gives others of the same ranges. `exact`
answers the same calls with plain torch in 64 bits.
"""
import math

import numpy as np
import torch

from chibillm_amd import ckv

PAGE = 16
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}

# Heads of one attention layer. "narrow": the KV shape of the benchmark's model (8 kv
# heads of 128, 16 query heads, rotary over the whole head). "wide": a layer with an
# output gate, 256-wide heads in groups of four and rotary on a quarter of the head.
NARROW = {"kv_heads": 8, "q_heads": 16, "head_dim": 128, "rotary": 128, "theta": 1e6, "gated": False}
WIDE = {"kv_heads": 2, "q_heads": 8, "head_dim": 256, "rotary": 64, "theta": 1e7, "gated": True}


def _case(op, heads, **more):
    return {"op": op, **heads, "dtype": "bf16", "layers": 1, **more}


def listed():
    return [
        # the smallest call: the default scheduler's four sequences early in a chat, one
        # layer of one decode step, where launches and round trips count
        dict(_case("decode", NARROW, rope=True, rows=4, low=64, high=512), name="decode 4 short rows"),
        # an ordinary serving batch: 32 sequences of mixed lengths
        dict(_case("decode", NARROW, rope=False, rows=32, low=256, high=4096), name="decode 32 rows"),
        # a full batch at long contexts, one layer of the benchmark's headline step
        dict(_case("decode", NARROW, rope=False, rows=128, low=1024, high=8192), name="decode 128 rows"),
        # one user with a long document: a single row has to fill the GPU
        dict(_case("decode", NARROW, rope=True, rows=1, low=32768, high=32768), name="decode one long row"),
        # pools in the storage type of the reference engine
        dict(_case("decode", NARROW, rope=False, rows=24, low=100, high=2500, dtype="f32"), name="decode f32 rows"),
        # a gated layer with wide heads, as hybrid models have them, in decode
        dict(_case("decode", WIDE, rope=True, rows=32, low=256, high=4096), name="decode wide heads"),
        # a whole decode step of an engine with a few live sequences: the batch goes up,
        # then 28 layers each rotate, append and attend
        dict(_case("step", NARROW, rope=True, rows=6, low=100, high=1500, layers=28), name="step of 28 layers"),
        # the middle of a long prompt: one sequence's next chunk, rotated, appended, attended
        dict(_case("prefill", NARROW, sequences=1, rows_low=512, rows_high=512, prefix=3000, shared=False), name="prefill one chunk"),
        # new prompts of mixed lengths batched together, nothing cached yet
        dict(_case("prefill", NARROW, sequences=9, rows_low=17, rows_high=450, prefix=0, shared=False, dtype="f16"), name="prefill new prompts"),
        # the largest: many sequences prefill behind one shared system prompt
        dict(_case("prefill", NARROW, sequences=64, rows_low=512, rows_high=512, prefix=2000, shared=True), name="prefill shared prefix"),
        # the gated wide layer in prefill
        dict(_case("prefill", WIDE, sequences=4, rows_low=300, rows_high=512, prefix=700, shared=False), name="prefill wide heads"),
        # a cached prefix packed for later and put back into other pages
        dict(_case("checkpoint", NARROW, tokens=2011, layers=28), name="checkpoint and restore"),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case of the listed ones' ranges; none costs more than the largest of its kind."""
    op = rng.choice(["decode"] * 4 + ["prefill"] * 3 + ["step", "checkpoint"])
    wide = op in ("decode", "prefill") and rng.random() < 0.3
    heads = dict(WIDE if wide else NARROW)
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16"] + ([] if wide else ["f32"]))
    if op == "checkpoint":
        return _case(op, heads, tokens=_log(rng, 64, 2011), layers=rng.choice([4, 12, 28]), dtype=dtype)
    if op == "step":
        low = _log(rng, 20, 200)
        return _case(op, heads, rope=True, rows=rng.randint(1, 6), low=low, high=low + _log(rng, 100, 1300), layers=28, dtype=rng.choice(["bf16", "f16"]))
    if wide:  # the same layer at other head counts of its kind
        heads["kv_heads"] = rng.choice([1, 2, 4])
        heads["q_heads"] = heads["kv_heads"] * rng.choice([2, 4])
        heads["gated"] = rng.random() < 0.7
    if op == "decode":
        rows = _log(rng, 1, 64 if wide else 128)
        most = max(64, min(32768, (60_000 if wide else 500_000 if dtype != "f32" else 120_000) // rows))
        high = _log(rng, 40, most)
        low = max(1, int(high * rng.uniform(0.05, 1.0)))
        rope = rng.random() < 0.5
        return _case(op, heads, rope=rope, rows=rows, low=low, high=high, dtype=dtype)
    sequences = _log(rng, 1, 4 if wide else 48)
    high = _log(rng, 9, 512)
    low = max(2, int(high * rng.uniform(0.1, 1.0)))
    # f32 products and, in the wide layer, long chunks are dear: shorter prefixes
    most = 700 if wide else 2000 if dtype != "f32" else 300
    prefix = rng.choice([0, _log(rng, 3, most)])
    if dtype == "f32":
        sequences = min(sequences, 6)
    return _case(op, heads, sequences=sequences, rows_low=low, rows_high=high, prefix=prefix, shared=prefix > 0 and sequences > 1 and rng.random() < 0.5, dtype=dtype)


# ---- shapes of a case (the same for every seed's work, positions drawn from the case alone) ----

def _lengths(case):
    """Context lengths of a decode batch, the new token included: spread evenly over
    [low, high] in a mixed order, so that every seed has the same work."""
    n, low, high = case["rows"], case["low"], case["high"]
    order = np.random.RandomState(n).permutation(n)
    return [int(x) for x in np.round(np.linspace(low, high, n))[order]] if n > 1 else [high]


def _chunks(case):
    """Rows of each sequence's chunk in a prefill."""
    n, low, high = case["sequences"], case["rows_low"], case["rows_high"]
    order = np.random.RandomState(n).permutation(n)
    return [int(x) for x in np.round(np.linspace(low, high, n))[order]] if n > 1 else [high]


def _pages(tokens):
    return -(-tokens // PAGE)


class _Batch:
    """Tables, positions and slots of a case's rows, over pages in an order drawn from the seed."""

    def __init__(self, case, seed):
        op = case["op"]
        if op == "checkpoint":
            spans, self.first = [case["tokens"]] * 2, []
        elif op == "prefill":
            spans = [case["prefix"] + n for n in _chunks(case)]
            self.first = [case["prefix"]] * len(spans)
        else:
            spans = _lengths(case)
            self.first = [n - 1 for n in spans]
        shared = case["prefix"] // PAGE if op == "prefill" and case["shared"] else 0
        need = shared + sum(_pages(n) - shared for n in spans)
        self.blocks = need + 7
        order = np.random.RandomState(seed % (1 << 32)).permutation(self.blocks).astype(np.uint32)
        self.tables, at = [], shared
        for n in spans:
            own = _pages(n) - shared
            self.tables.append(np.concatenate([order[:shared], order[at:at + own]]))
            at += own
        self.spans = spans
        if op == "checkpoint":
            return
        counts = [n - f for n, f in zip(spans, self.first)]
        self.counts = counts
        self.seq = np.repeat(np.arange(len(spans)), counts)
        self.positions = np.concatenate([np.arange(f, f + c) for f, c in zip(self.first, counts)]).astype(np.uint32)
        starts = np.concatenate([[0], np.cumsum([t.size for t in self.tables])[:-1]])
        self.flat = np.concatenate(self.tables)
        self.offsets = starts[self.seq].astype(np.uint32)
        self.lengths = np.array([t.size for t in self.tables], np.uint32)[self.seq]
        page = self.flat[self.offsets + self.positions // PAGE]
        self.slots = (page.astype(np.uint64) * PAGE + self.positions % PAGE).astype(np.uint32)


def _tensors(case, seed, batch):
    """The case's device arrays, from the seed alone: the pool's pages and each layer's new rows."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt, layers = DTYPES[case["dtype"]], case["layers"]
    f, qf = case["kv_heads"] * case["head_dim"], case["q_heads"] * case["head_dim"]

    def randn(*shape):
        return torch.randn(*shape, generator=g, dtype=dt, device="cuda")

    t = {"keys": randn(layers, batch.blocks * PAGE, f), "values": randn(layers, batch.blocks * PAGE, f)}
    if case["op"] != "checkpoint":
        rows = len(batch.positions)
        t["k"], t["v"], t["q"] = randn(layers, rows, f), randn(layers, rows, f), randn(layers, rows, qf)
        t["gate"] = randn(layers, rows, qf) if case["gated"] else None
    return t


def prepare(case, seed):
    batch = _Batch(case, seed)
    t = _tensors(case, seed, batch)
    ctx = ckv.Context(0, stream=torch.cuda.current_stream())
    pool = ckv.Pool(ctx, case["layers"], batch.blocks, PAGE, case["kv_heads"], case["head_dim"],
                    DTYPES[case["dtype"]], t["keys"], t["values"])
    state = {"case": case, "batch": batch, "ctx": ctx, "pool": pool, "scale": 1.0 / math.sqrt(case["head_dim"]), **t}
    if case["op"] == "checkpoint":
        f = case["kv_heads"] * case["head_dim"]
        state["packed"] = [torch.empty(case["layers"], case["tokens"], f, dtype=t["keys"].dtype, device="cuda") for _ in range(2)]
        return state
    state["out"] = torch.empty_like(t["q"])
    if case["op"] == "step":
        # the engine's arena of sequence tables, as it stands before the step
        width = max(x.size for x in batch.tables) + 8
        pool.reserve_sequences(len(batch.tables), width)
        n = [x.size for x in batch.tables]
        pool.update_sequences(np.repeat(np.arange(len(n)), n), np.concatenate([np.arange(x) for x in n]), batch.flat, np.arange(len(n)), n)
        state["items"] = (np.arange(len(n), dtype=np.uint32), np.array(batch.first, np.uint32), np.ones(len(n), np.uint32))
    else:
        pool.upload(batch.flat, batch.offsets, batch.lengths, batch.positions, batch.slots)
    if case["op"] == "prefill":
        state["rotated"] = torch.empty_like(t["q"])
    return state


def _layer_decode(s, layer):
    c, pool = s["case"], s["pool"]
    k, v, q, out = s["k"][layer], s["v"][layer], s["q"][layer], s["out"][layer]
    gate = None if s["gate"] is None else s["gate"][layer]
    if c["rope"]:
        pool.rope_append_decode(layer, k, v, q, c["q_heads"], s["scale"], c["theta"], out, rotary_dim=c["rotary"], gate=gate)
    elif gate is not None:
        pool.append_decode_gated(layer, k, v, q, c["q_heads"], s["scale"], gate, out)
    else:
        pool.append_decode(layer, k, v, q, c["q_heads"], s["scale"], out)


def run(s):
    c, pool = s["case"], s["pool"]
    if c["op"] == "checkpoint":
        batch = s["batch"]
        pool.checkpoint_pack(batch.tables[0], c["tokens"], *s["packed"])
        pool.checkpoint_unpack(batch.tables[1], c["tokens"], *s["packed"])
        return {"packed_keys": s["packed"][0], "packed_values": s["packed"][1], "keys": s["keys"], "values": s["values"]}
    if c["op"] == "step":
        pool.upload_batch(*s["items"])
    if c["op"] == "prefill":
        pool.rope(s["q"][0], s["rotated"][0], c["q_heads"], c["theta"], c["rotary"])
        pool.rope_append(0, s["k"][0], s["v"][0], c["theta"], c["rotary"])
        if s["gate"] is not None:
            pool.attention_gated(0, s["rotated"][0], c["q_heads"], s["scale"], s["gate"][0], s["out"][0])
        else:
            pool.attention(0, s["rotated"][0], c["q_heads"], s["scale"], s["out"][0])
    else:
        for layer in range(c["layers"]):
            _layer_decode(s, layer)
    return {"out": s["out"], "keys": s["keys"], "values": s["values"]}


def work(case):
    """Bytes read and written once, and the products of q.k and p.v."""
    size = 4 if case["dtype"] == "f32" else 2
    f, qf = case["kv_heads"] * case["head_dim"], case["q_heads"] * case["head_dim"]
    if case["op"] == "checkpoint":
        return {"bytes": 2 * 4.0 * case["layers"] * case["tokens"] * f * size, "flops": 0.0}
    if case["op"] == "prefill":
        counts, prefix = _chunks(case), case["prefix"]
        held = prefix * (1 if case["shared"] else len(counts))
        pairs = sum(n * prefix + n * (n + 1) / 2 for n in counts)
    else:
        lengths = _lengths(case)
        counts, held, pairs = [1] * len(lengths), sum(lengths) - len(lengths), sum(lengths)
    rows = sum(counts)
    # cached keys and values read; the new rows read and written; queries, gate and output
    moved = held * 2 * f + rows * 4 * f + rows * qf * (3 if case["gated"] else 2)
    return {"bytes": float(case["layers"] * moved * size), "flops": 4.0 * case["layers"] * pairs * qf}


def tolerance(case):
    if case["op"] == "checkpoint":
        return "exact"
    # f32: sums in another order, and exponentials a few units off. 16-bit: the output's
    # rounding and, on matrix units, the probabilities'; rotated rows are rounded too
    # (against 64 bits the 16-bit calls are 1.6e-3 to 2.9e-3 off in bf16, 3.3e-4 in f16).
    return {"f32": {"rel": 1e-5, "max": 2e-4}, "f16": {"rel": 1.5e-3, "max": 1e-2}, "bf16": {"rel": 1e-2, "max": 6e-2}}[case["dtype"]]


# ---- the same calls in 64 bits ----

def _rotate(x, positions, case):
    """Rotary embedding of [rows, heads * head_dim] in 64 bits."""
    rows, d, r = x.shape[0], case["head_dim"], case["rotary"]
    x = x.double().reshape(rows, -1, d)
    j = torch.arange(r // 2, dtype=torch.float64, device=x.device)
    angle = positions[:, None].double() * case["theta"] ** (-2.0 * j / r)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., :r // 2], x[..., r // 2:r]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., r:]], -1).reshape(rows, -1)


def exact(case, seed):
    batch = _Batch(case, seed)
    t = _tensors(case, seed, batch)
    if case["op"] == "checkpoint":
        n = case["tokens"]

        def slots_of(table):
            p = torch.arange(n, device="cuda")
            return torch.from_numpy(table.astype(np.int64)).cuda()[p // PAGE] * PAGE + p % PAGE

        source, target = slots_of(batch.tables[0]), slots_of(batch.tables[1])
        packed = [t[x][:, source].double() for x in ("keys", "values")]
        keys, values = t["keys"].double(), t["values"].double()
        keys[:, target], values[:, target] = packed
        return {"packed_keys": packed[0], "packed_values": packed[1], "keys": keys, "values": values}
    h, d = case["kv_heads"], case["head_dim"]
    group, scale = case["q_heads"] // h, 1.0 / math.sqrt(d)
    positions = torch.from_numpy(batch.positions.astype(np.int64)).cuda()
    slots = torch.from_numpy(batch.slots.astype(np.int64)).cuda()
    rope = case["op"] == "prefill" or case["rope"]
    keys, values = t["keys"].double(), t["values"].double()
    out = torch.empty(t["q"].shape, dtype=torch.float64, device="cuda")
    for layer in range(case["layers"]):
        k, q = t["k"][layer].double(), t["q"][layer].double()
        if rope:
            k, q = _rotate(k, positions, case), _rotate(q, positions, case)
        keys[layer, slots], values[layer, slots] = k, t["v"][layer].double()
        row = 0
        for table, first, count in zip(batch.tables, batch.first, batch.counts):
            p = torch.arange(first + count, device="cuda")
            at = torch.from_numpy(table.astype(np.int64)).cuda()[p // PAGE] * PAGE + p % PAGE
            ks = keys[layer, at].reshape(-1, h, d).permute(1, 2, 0).contiguous()  # [h, d, tokens]
            vs = values[layer, at].reshape(-1, h, d).permute(1, 0, 2).contiguous()
            qs = q[row:row + count].reshape(count, h, group, d).permute(1, 2, 0, 3).reshape(h, group * count, d)
            s = torch.bmm(qs.contiguous(), ks) * scale
            hidden = p[None, :] > (first + torch.arange(count, device="cuda"))[:, None]
            s = s.reshape(h, group, count, -1).masked_fill(hidden, -math.inf).softmax(-1).reshape(h, group * count, -1)
            o = torch.bmm(s, vs).reshape(h, group, count, d).permute(2, 0, 1, 3)
            out[layer, row:row + count] = o.reshape(count, -1)
            row += count
        if t["gate"] is not None:
            out[layer] *= torch.sigmoid(t["gate"][layer].double())
    return {"out": out, "keys": keys, "values": values}
