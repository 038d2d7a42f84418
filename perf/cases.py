"""The embedding lookups that are timed: which calls, at which sizes, on which values.

Every case is one call (or one forward and backward) of a public entry point,
as a program that serves or trains an embedding model makes it:

  rows        pynve.torch.NVEmbedding over a table in HBM, inference: a row per key
  bags        pynve.torch.NVEmbeddingBag over a table in HBM, inference: a row per bag
  multi       nve_amd_find_and_pool_multi: the jagged bags of several tables in one call
  quant_rows  nve_layer_lookup_pooled, Concatenate, rowwise-quantized rows: a dequantized row per key
  quant_bags  nve_layer_lookup_pooled, rowwise-quantized rows: a row per bag
  train_rows  NVEmbedding built for training: forward, then the sparse gradient of the table
  train_bags  NVEmbeddingBag built for training: forward, then the sparse gradient of the table
  uvm_rows    NVEmbedding over a host-resident table with a warmed cache in HBM
  uvm_bags    NVEmbeddingBag over a host-resident table with a warmed cache in HBM

Keys are Zipf distributed over the rows (alpha 0: uniform), ranks spread over
the table; jagged bags have Poisson lengths.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "nv-embedding-cache_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

# name -> (type id of the C ABI, bytes of scale and offset after the values)
_QUANT = {"qi8_f32": (7, 4), "qi8_f16": (8, 2), "qu8_f32": (9, 8), "qu8_f16": (10, 4),
          "xi8a_f32": (32, 8), "xe4m3_f32": (33, 4)}
_TORCH = {"f32": torch.float32, "f16": torch.float16}
_SIZE = {"f32": 4, "f16": 2}
_POOL = {"concat": 0, "sum": 1, "mean": 2, "wsum": 3, "wmean": 4}
_INT64_KEYS, _CSR = 1, 1


def _case(op, **fields):
    """Every case has the same fields, so that a new one is a change of values only."""
    c = {"op": op, "rows": 1000000, "dim": 128, "dtype": "f16", "out": "", "keys": 0, "bags": 0,
         "mean_len": 0, "jagged": False, "mode": "sum", "alpha": 1.05, "tables": 1, "cache_mib": 0}
    c.update(fields)
    if not c["out"]:
        c["out"] = c["dtype"]
    return c


def listed():
    named = {
        # one request of an online service: a few hundred ids of one feature
        "rows_request": _case("rows", rows=1000000, dim=64, dtype="f32", keys=512, alpha=0.0),
        # a whole batch of single-valued features from a table far beyond the caches
        "rows_batch": _case("rows", rows=50000000, keys=262144),
        # a batch of short fixed bags (4,096 samples of 8 ids)
        "bags_short": _case("bags", rows=1000000, dim=64, dtype="f32", bags=4096, mean_len=8, alpha=0.0),
        # long histories: few bags, a thousand ids each
        "bags_long": _case("bags", rows=50000000, bags=256, mean_len=1024),
        # a ranking model's jagged, weighted feature whose width is no power of two
        "bags_odd": _case("bags", rows=4000000, dim=100, bags=16384, mean_len=30, jagged=True, mode="wmean",
                          alpha=1.1),
        # all sparse features of a recommender's batch at once
        "multi_26": _case("multi", rows=40000000, out="f32", bags=8192, mean_len=20, jagged=True, mode="wmean",
                          alpha=1.1, tables=26),
        # a quantized table served row by row
        "quant_rows": _case("quant_rows", rows=100000000, dim=256, dtype="xi8a_f32", out="f16", keys=131072),
        # a quantized table served as pooled jagged features
        "quant_bags": _case("quant_bags", rows=20000000, dim=128, dtype="qi8_f32", out="f32", bags=16384,
                            mean_len=30, jagged=True, alpha=1.1),
        # a training step over a sequence or an id feature: a gradient row per distinct id
        "train_rows": _case("train_rows", rows=1000000, dim=64, dtype="f32", keys=32768),
        # a training step over long bags
        "train_bags": _case("train_bags", rows=50000000, bags=256, mean_len=1024),
        # a table too large for HBM, most ids in the cache: rows for a sequence model
        "uvm_rows": _case("uvm_rows", rows=2000000, keys=65536, alpha=1.2, cache_mib=128),
        # the same for pooled jagged features, nearly all ids in the cache
        "uvm_bags": _case("uvm_bags", rows=2000000, bags=8192, mean_len=20, jagged=True, alpha=1.2, cache_mib=400),
    }
    return [dict(c, name=n) for n, c in named.items()]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A row width: half of them multiples of 8, as models mostly have, the others any."""
    d = _log(rng, lo, hi)
    return max(lo, d // 8 * 8) if rng.random() < 0.5 else d


def _draw(rng):
    op = rng.choice(["rows", "bags", "multi", "quant_rows", "quant_bags", "train_rows", "train_bags",
                     "uvm_rows", "uvm_bags"])
    quant, uvm, train = op.startswith("quant"), op.startswith("uvm"), op.startswith("train")
    dtype = rng.choice(list(_QUANT)) if quant else rng.choice(["f32", "f16"])
    out = dtype
    if quant:
        out = rng.choice(["f32", "f16"]) if dtype[0] == "x" else dtype[-3:]
    elif op == "multi":
        out = rng.choice(["f32", "f16"])
    c = _case(op, dtype=dtype, out=out, alpha=rng.choice([0.0, 1.05, 1.1, 1.2]),
              rows=_log(rng, 50000, 2000000) if uvm else _log(rng, 10000, 20000000))
    if uvm and c["alpha"] == 0.0:
        c["alpha"] = 1.2
    c["dim"] = _width(rng, 8, 256 if train or uvm or op == "multi" else 768)
    if quant:  # quantized rows have an even width
        c["dim"] = max(16, c["dim"] // 2 * 2)
    if op.endswith("rows"):
        c["keys"] = _log(rng, 64, 65536 if uvm else 262144)
    else:
        c["jagged"] = rng.random() < 0.7
        c["mode"] = rng.choice(["sum", "mean", "wsum", "wmean"])
        c["tables"] = _log(rng, 2, 40) if op == "multi" else 1
        c["mean_len"] = _log(rng, 2, 64 if uvm or op == "multi" else 1024)
        most = (65536 if uvm else 262144 if train else 524288) // c["mean_len"]
        if op == "multi":
            most = 2000000 // (c["mean_len"] * c["tables"])
        c["bags"] = _log(rng, 16, max(32, min(16384, most)))
    if uvm:
        c["cache_mib"] = max(8, int(c["rows"] * _row_bytes(c) * rng.uniform(0.1, 0.8)) >> 20)
    return c


def draw(rng):
    """A case of the same kinds: any type, option and width, from a handful of keys to a full batch."""
    most = max(work(c)["bytes"] for c in listed())
    while True:
        c = _draw(rng)
        table = c["rows"] * _row_bytes(c)
        if c["tables"] > 1:  # log-uniform row counts: the expected total
            table *= c["tables"] / math.log(c["rows"] / 1e3) / 2
        if work(c)["bytes"] <= most and table <= (1 << 30 if c["op"].startswith("uvm") else 13 << 30):
            return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _meta(c):
    return _QUANT[c["dtype"]][1] if c["dtype"] in _QUANT else 0


def _row_bytes(c):
    return c["dim"] + _meta(c) if c["dtype"] in _QUANT else c["dim"] * _SIZE[c["dtype"]]


def _cardinalities(c, seed):
    """Rows of each table: one table has `rows`; several are log-uniform from 1e3 to `rows`."""
    if c["tables"] == 1:
        return [c["rows"]]
    r = np.random.default_rng([seed, 11])
    return [int(v) for v in np.exp(r.uniform(math.log(1e3), math.log(c["rows"]), c["tables"]))]


def _zipf(n, rows, alpha, gen, moved=None):
    """n row ids: ranks of a power law over the rows (uniform for alpha 0), spread over the table.

    With `moved`, the ranks are the same for every seed, in an order and on
    rows that `moved` (another generator) gives, so that every seed has the
    same number of distinct rows."""
    x = torch.rand(n, device="cuda", dtype=torch.float64, generator=gen)
    if alpha == 0.0:
        rank = (x * rows).long().clamp_(0, rows - 1)
    else:
        g = 1.0 - alpha
        rank = (x * (float(rows) ** g - 1.0) + 1.0).pow(1.0 / g).long().clamp_(1, rows) - 1
    shift = 12345
    if moved is not None:
        rank = rank[torch.randperm(n, device="cuda", generator=moved)]
        shift = torch.randint(0, rows, (1,), device="cuda", generator=moved)
    step = 2654435761  # a prime above every row count here: the map below moves each rank to a row of its own
    return (rank * step + shift) % rows


def _float_table(rows, dim, dtype, gen):
    t = torch.empty((rows, dim), device="cuda", dtype=_TORCH[dtype])
    _fill(t, gen)
    return t


def _fill(t, gen):
    step = max(1, (1 << 28) // t.shape[1])
    for r in range(0, t.shape[0], step):
        t[r:r + step].normal_(0.0, 0.02, generator=gen)


def _quant_table(c, gen):
    """Stored rows as bytes: values, then scale (log-uniform 1e-3 to 1e-1) and offset (N(0, 0.01))."""
    rows, dim, meta, dt = c["rows"], c["dim"], _meta(c), c["dtype"]
    half = dt.endswith("f16")
    t = torch.empty((rows, dim + meta), device="cuda", dtype=torch.uint8)
    step = max(1, (1 << 28) // dim)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        q = torch.randint(0, 256, (n, dim), device="cuda", dtype=torch.uint8, generator=gen)
        if dt == "xe4m3_f32":
            q -= ((q & 0x7F) == 0x7F).to(torch.uint8)  # no NaN codes
        elif dt[:3] == "qi8" or dt[:3] == "xi8":
            q += (q == 128).to(torch.uint8)  # -127 .. 127
        t[r:r + n, :dim] = q
        u = torch.rand((n, 1), device="cuda", generator=gen)
        m = [torch.exp(math.log(1e-3) + u * math.log(1e2))]
        if meta // (2 if half else 4) == 2:
            m.append(torch.randn((n, 1), device="cuda", generator=gen) * 0.01)
        t[r:r + n, dim:] = torch.cat([v.to(torch.float16 if half else torch.float32).view(torch.uint8) for v in m], 1)
    return t


def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 16 + what)
    return g


def _inputs(c, seed):
    """Keys, offsets (bags only), weights (weighted modes only) and table row counts."""
    cards = _cardinalities(c, seed)
    kg, lg, wg, moved = _gen(seed, 1), _gen(seed, 2), _gen(seed, 3), None
    if c["op"].startswith("train"):  # gradients of the same number of rows for every seed
        kg, lg, moved = _gen(0, 1), _gen(0, 2), _gen(seed, 1)
    if c["bags"] == 0:
        keys = _zipf(c["keys"], c["rows"], c["alpha"], kg, moved)
        return {"cards": cards, "offsets": None, "weights": None, "keys": keys}
    bags = c["bags"] * len(cards)
    lens = torch.full((bags,), float(c["mean_len"]), device="cuda")
    if c["jagged"]:
        lens = torch.poisson(lens, generator=lg).clamp_(0, 5 * c["mean_len"])
    offsets = torch.zeros(bags + 1, dtype=torch.int64, device="cuda")
    offsets[1:] = torch.cumsum(lens.long(), 0)
    ends = offsets[:: c["bags"]].tolist()
    keys = torch.cat([_zipf(e - s, r, c["alpha"], kg, moved) for s, e, r in zip(ends, ends[1:], cards)])
    weights = None
    if c["mode"][0] == "w":
        wt = torch.float32 if c["op"] in ("multi", "quant_bags") else _TORCH[c["dtype"]]
        weights = torch.rand(keys.numel(), device="cuda", generator=wg).to(wt)
    return {"cards": cards, "offsets": offsets, "weights": weights, "keys": keys}


def _tables(c, seed, cards):
    g = _gen(seed, 4)
    if c["dtype"] in _QUANT:
        return [_quant_table(c, g)]
    return [_float_table(r, c["dim"], c["dtype"], g) for r in cards]


def _out_grad(c, seed, rows):
    return torch.empty((rows, c["dim"]), device="cuda", dtype=_TORCH[c["dtype"]]).normal_(0.0, 1.0, generator=_gen(seed, 5))


# ---------------------------------------------------------------------------
# the program's state and one pass
# ---------------------------------------------------------------------------
class _QuantLayer:
    """A GPU layer over quantized rows through the C ABI, with its execution context."""

    def __init__(self, c, table):
        from pynve import _lib

        self.lib, self.table = _lib, table
        cfg = _lib.load().nve_gpu_embedding_layer_config_default()
        cfg.layer_name, cfg.device_id = b"quant", torch.cuda.current_device()
        cfg.embedding_table, cfg.num_embeddings = table.data_ptr(), table.shape[0]
        cfg.embedding_width_in_bytes, cfg.value_dtype = table.shape[1], _QUANT[c["dtype"]][0]
        self.layer, self.ctx = ctypes.c_void_p(), ctypes.c_void_p()
        _lib.call("nve_gpu_embedding_layer_create", ctypes.byref(self.layer), _INT64_KEYS, ctypes.byref(cfg), None)
        _lib.call("nve_layer_create_execution_context", self.layer, ctypes.byref(self.ctx),
                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), None, None, None)

    def __del__(self):
        if getattr(self, "ctx", None) and self.ctx.value:
            self.lib.load().nve_context_destroy(self.ctx)
        if getattr(self, "layer", None) and self.layer.value:
            self.lib.load().nve_layer_destroy(self.layer)


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _module(c, seed):
    from pynve.torch import nve_layers as nl

    uvm = c["op"].startswith("uvm")
    kw = {"optimize_for_training": c["op"].startswith("train")}
    kind = nl.LayerType.GPULayer
    if uvm:
        kind = nl.LayerType.LinearUVM
        kw["gpu_cache_size"] = c["cache_mib"] << 20
    if c["bags"]:
        m = nl.NVEmbeddingBag(c["rows"], c["dim"], _TORCH[c["dtype"]], kind, c["mode"].lstrip("w"), **kw)
    else:
        m = nl.NVEmbedding(c["rows"], c["dim"], _TORCH[c["dtype"]], kind, **kw)
    if not uvm:
        _fill(m.weight.data, _gen(seed, 4))
        return m
    table = _tables(c, seed, [c["rows"]])[0]
    m.weight.data.copy_(table)
    for b in range(10):  # warmed with ten batches of the same traffic
        keys = _zipf(max(1, c["keys"] or c["bags"] * c["mean_len"]), c["rows"], c["alpha"], _gen(seed, 6 + b))
        m.insert(keys, table[keys], 0)
    torch.cuda.synchronize()
    return m


def prepare(case, seed):
    c, s = case, _inputs(case, seed)
    s["case"] = c
    if c["op"].startswith("quant"):
        s["layer"] = _QuantLayer(c, _tables(c, seed, s["cards"])[0])
        rows = c["bags"] or c["keys"]
        s["output"] = torch.empty((rows, c["dim"]), device="cuda", dtype=_TORCH[c["out"]])
    elif c["op"] == "multi":
        s["tables"] = _tables(c, seed, s["cards"])
        s["table_ptrs"] = (ctypes.c_void_p * c["tables"])(*[t.data_ptr() for t in s["tables"]])
        s["table_rows"] = (ctypes.c_int64 * c["tables"])(*s["cards"])
        s["output"] = torch.empty((c["bags"], c["tables"], c["dim"]), device="cuda", dtype=_TORCH[c["out"]])
    else:
        s["module"] = _module(c, seed)
        if c["op"].startswith("train"):
            s["grad"] = _out_grad(c, seed, c["bags"] or c["keys"])
    return s


def run(state):
    s, c = state, state["case"]
    op = c["op"]
    if op.startswith("quant"):
        q, out, off, w = s["layer"], s["output"], s["offsets"], s["weights"]
        pool = _POOL["concat"] if op == "quant_rows" else _POOL[c["mode"]]
        q.lib.call("nve_layer_lookup_pooled", q.layer, q.ctx, s["keys"].numel(), _ptr(s["keys"]), _ptr(out),
                   out.shape[1] * out.element_size(), None, pool, _CSR, _ptr(off),
                   0 if off is None else off.numel(), 0, _ptr(w), 0 if w is None else 1,
                   1 if c["out"] == "f32" else 3, None)
        return out
    if op == "multi":
        from pynve import _lib

        out, w = s["output"], s["weights"]
        _lib.call("nve_amd_find_and_pool_multi", _INT64_KEYS, c["tables"], s["table_ptrs"], s["table_rows"],
                  _row_bytes(c), 1 if c["dtype"] == "f32" else 3, c["bags"], s["keys"].numel(), _ptr(s["keys"]),
                  _ptr(s["offsets"]), _ptr(w), 0 if w is None else 1, _POOL[c["mode"]],
                  1 if c["out"] == "f32" else 3, _ptr(out),
                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        return out
    m = s["module"]
    if op.startswith("train"):
        out = m(s["keys"], s["offsets"], s["weights"]) if c["bags"] else m(s["keys"])
        (g,) = torch.autograd.grad(out, m.weight, s["grad"])
        return {"out": out, "grad_rows": g._indices()[0], "grad": g._values()}
    with torch.no_grad():
        return m(s["keys"], s["offsets"], s["weights"]) if c["bags"] else m(s["keys"])


# ---------------------------------------------------------------------------
# what a pass cannot do without, and what it computes
# ---------------------------------------------------------------------------
def _distinct(n, rows, alpha):
    """Expected number of distinct rows among n keys."""
    if alpha == 0.0:
        return rows * -math.expm1(n * math.log1p(-1.0 / rows)) if rows > 1 else 1.0
    edge = np.unique(np.round(np.geomspace(1, rows + 1, 20000)))
    g = 1.0 - alpha
    mass = np.diff((edge ** g - 1.0) / (float(rows) ** g - 1.0))
    size = np.diff(edge)
    each = np.clip(mass / size, 0.0, 1.0 - 1e-12)
    return float(np.sum(size * -np.expm1(n * np.log1p(-each))))


def work(case):
    c = case
    n = c["keys"] or c["bags"] * c["mean_len"]
    cards = _cardinalities(c, 0)
    seen = sum(_distinct(n, r, c["alpha"]) for r in cards)
    n *= len(cards)
    out_rows = n if c["bags"] == 0 else c["bags"] * len(cards)
    out = out_rows * c["dim"] * _SIZE[c["out"]]
    side = 8 * n
    if c["bags"]:
        side += 8 * (out_rows + 1)
        if c["mode"][0] == "w":
            side += n * (4 if c["op"] in ("multi", "quant_bags") else _SIZE[c["dtype"]])
    total = side + seen * _row_bytes(c) + out
    if c["op"].startswith("train"):  # the gradient of the output in, ids and gradient rows out
        total += out + seen * (8 + _row_bytes(c))
    flops = n * c["dim"] * (2.0 if c["op"].startswith("train") else 1.0)
    return {"bytes": float(total), "flops": float(flops)}


def tolerance(case):
    """Plain rows are copies.  Sums are fp32, rounded once to the output type."""
    c = case
    if c["op"] in ("rows", "uvm_rows"):
        return "exact"
    if c["out"] == "f16":
        return {"rel": 8e-4, "max": 4e-3}
    return {"rel": 1e-6, "max": 2e-5}


def _e4m3_values():
    return torch.arange(256, dtype=torch.uint8).view(torch.float8_e4m3fn).to(torch.float64).cuda()


def _values64(c, table, keys):
    """The rows of `keys` in 64 bits, dequantized where they are stored as bytes."""
    rows = table[keys]
    if c["dtype"] not in _QUANT:
        return rows.double()
    dim, meta, dt = c["dim"], _meta(c), c["dtype"]
    ft = torch.float16 if dt.endswith("f16") else torch.float32
    m = rows[:, dim:].contiguous().view(ft).double()
    q = rows[:, :dim]
    if dt == "xe4m3_f32":
        x = _e4m3_values()[q.long()]
    else:
        x = (q if dt[:3] == "qu8" else q.contiguous().view(torch.int8)).double()
    x = x * m[:, :1]
    return x + m[:, 1:] if m.shape[1] == 2 else x


def _bag_weights(c, x, bag, bags):
    """The factor of each key in its bag: 1 or its weight, over the bag's length or weight sum for means."""
    w = torch.ones(bag.numel(), device="cuda", dtype=torch.float64) if x["weights"] is None else x["weights"].double()
    if c["mode"].endswith("mean"):
        d = torch.zeros(bags, device="cuda", dtype=torch.float64).index_add_(0, bag, w)[bag]
        w = torch.where(d == 0, torch.zeros_like(w), w / d)
    return w


def _pool64(c, x, tables):
    bags = x["offsets"].numel() - 1
    bag = torch.repeat_interleave(torch.arange(bags, device="cuda"), torch.diff(x["offsets"]))
    w = _bag_weights(c, x, bag, bags)
    out = torch.zeros((bags, c["dim"]), device="cuda", dtype=torch.float64)
    ends = x["offsets"][:: c["bags"]].tolist()
    for table, s, e in zip(tables, ends, ends[1:]):
        for i in range(s, e, 1 << 19):
            j = slice(i, min(e, i + (1 << 19)))
            out.index_add_(0, bag[j], _values64(c, table, x["keys"][j]) * w[j, None])
    return out, bag, w


def exact(case, seed):
    c, x = case, _inputs(case, seed)
    tables = _tables(c, seed, x["cards"])
    if c["bags"] == 0:
        out, bag, w = _values64(c, tables[0], x["keys"]), None, None
    else:
        out, bag, w = _pool64(c, x, tables)
    if c["op"] == "multi":
        return out.view(c["tables"], c["bags"], c["dim"]).transpose(0, 1).contiguous()
    if not c["op"].startswith("train"):
        return out
    rows, where = torch.unique(x["keys"], return_inverse=True)
    g = _out_grad(c, seed, c["bags"] or c["keys"]).double()
    grad = torch.zeros((rows.numel(), c["dim"]), device="cuda", dtype=torch.float64)
    for i in range(0, where.numel(), 1 << 19):
        j = slice(i, i + (1 << 19))
        grad.index_add_(0, where[j], g[j] if bag is None else g[bag[j]] * w[j, None])
    return {"out": out, "grad_rows": rows, "grad": grad}
