"""The work that a program using this library has it do, as cases to time.

A table here is a few columns that are stored together, each with the tree
its data calls for; columns are resident in HBM, as the library's callers
keep them, and every pass goes through the Python package's public classes.
Four tables of data:

* ``int``    the four int32 columns of the single-scheme workload: event
  times (delta, then FL), a step function (RLE, both outputs FL), codes of a
  50-value dictionary, and measurements with 1% outliers (patch, both sides
  FL);
* ``float``  price walks: float64 and float32 through GFC, float64 as
  integers through delta and FL, float32 through scale, delta and FL;
* ``mixed``  the narrower and wider types: int64 times in microseconds,
  int16 sensor levels, int8 states that hold for a while, a mostly constant
  int16 column and long-tailed int32 volumes through a nested dictionary;
* ``batch``  many columns of very different lengths compressed by one call.

Outputs are the blobs, the decoded columns and the chosen trees: all of them
bytes or whole numbers, so every tolerance is "exact".  A blob's length depends
on the data; it is returned as its length and a view of two rows of a fixed
length, its first and its last bytes, which together cover it.
"""
from __future__ import annotations

import math

import torch

import gputimeseriescompressionoptimizer_amd as g
from gputimeseriescompressionoptimizer_amd.train_planner import WEIGHTS

DEVICE = "cuda:0"
_ctx = None


def context() -> g.Context:
    """The program's one context: a stream and a caching allocator."""
    global _ctx
    if _ctx is None:
        _ctx = g.Context(0)
    return _ctx


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # One block of 10,000 readings written and read back: the sample size of
        # the reference's optimizer, where launches and read-backs are all.
        {"name": "int_roundtrip_10k", "kind": "table", "table": "int", "dir": "roundtrip", "rows": 10_000},
        # The column API's default batch (a million rows), not a multiple of anything.
        {"name": "int_encode_1m", "kind": "table", "table": "int", "dir": "encode", "rows": 1_000_003},
        {"name": "int_decode_1m", "kind": "table", "table": "int", "dir": "decode", "rows": 1_000_003},
        # The single-scheme workload at its full size.
        {"name": "int_encode_64m", "kind": "table", "table": "int", "dir": "encode", "rows": 67_108_864},
        {"name": "int_decode_64m", "kind": "table", "table": "int", "dir": "decode", "rows": 67_108_864},
        # Price history, 32M quotes per column.
        {"name": "float_encode_32m", "kind": "table", "table": "float", "dir": "encode", "rows": 33_554_393},
        {"name": "float_decode_32m", "kind": "table", "table": "float", "dir": "decode", "rows": 33_554_393},
        # A sensor log of narrow and wide columns, written and read back.
        {"name": "mixed_roundtrip_5m", "kind": "table", "table": "mixed", "dir": "roundtrip", "rows": 5_000_011},
        # A table of 48 columns of 4K..4M rows compressed by one call.
        {"name": "batch_48_columns", "kind": "batch", "columns": 48, "max_rows": 4_000_000},
        # A column that arrives in parts through the adaptive optimizer, which
        # plans on the first part and every tenth; its data changes half-way.
        {"name": "optimizer_12_parts", "kind": "optimizer", "parts": 12, "rows": 10_007},
        # Blocks planned by the learned planner, then compressed with its tree.
        {"name": "learned_16_blocks", "kind": "learned", "blocks": 16, "rows": 65_537},
        # Range queries and point look-ups in compressed columns.
        {"name": "access_32m", "kind": "access", "rows": 33_554_393, "ranges": 8, "range_rows": 65_537,
         "fetch": 1_000_003},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["table", "table", "table", "batch", "optimizer", "learned", "access"])
    if kind == "table":
        table = rng.choice(["int", "int", "float", "mixed"])
        top = {"int": 67_108_864, "float": 33_554_393, "mixed": 8_000_000}[table]
        return {"kind": kind, "table": table, "dir": rng.choice(["encode", "decode", "roundtrip"]),
                "rows": _log_uniform(rng, 1_000, top // 2 if table != "mixed" else top)}
    if kind == "batch":
        return {"kind": kind, "columns": rng.randint(8, 60), "max_rows": _log_uniform(rng, 100_000, 4_000_000)}
    if kind == "optimizer":
        return {"kind": kind, "parts": rng.randint(3, 14), "rows": _log_uniform(rng, 10_000, 200_000)}
    if kind == "learned":
        return {"kind": kind, "blocks": rng.randint(4, 24), "rows": _log_uniform(rng, 10_000, 1_048_576)}
    rows = _log_uniform(rng, 1_000_000, 33_554_393)
    return {"kind": kind, "rows": rows, "ranges": rng.randint(1, 12), "range_rows": _log_uniform(rng, 1_000, 500_000),
            "fetch": _log_uniform(rng, 1_000, 2_000_000)}


# --------------------------------------------------------------------- data
def _uniform(n, gen):
    """float32 in (0, 1]."""
    return 1.0 - torch.rand(n, generator=gen, device=DEVICE)


def _geometric(n, p, gen):
    return torch.floor(torch.log(_uniform(n, gen)) / math.log1p(-p)).to(torch.int64) + 1


def _choice(n, weights, gen):
    cdf = torch.tensor(weights, dtype=torch.float64).cumsum(0)
    cdf = (cdf / cdf[-1]).to(DEVICE, torch.float32)
    return torch.searchsorted(cdf, torch.rand(n, generator=gen, device=DEVICE)).clamp_(max=len(weights) - 1)


def _zipf_weights(k, s):
    return [1.0 / (i + 1) ** s for i in range(k)]


def timestamps(n, gen, p=0.3):
    return (1_400_000_000 + _geometric(n, p, gen).cumsum(0)).to(torch.int32)


def times_us(n, gen):
    return 1_400_000_000_000_000 + (_geometric(n, 0.001, gen)).cumsum(0)


def _runs(n, mean_run, values, gen):
    """`values` repeated over geometric run lengths, cut to n rows."""
    k = int(n / mean_run * 1.2) + 64
    lens = _geometric(k, 1.0 / mean_run, gen)
    x = torch.repeat_interleave(values(k), lens)
    while x.numel() < n:
        x = torch.cat([x, torch.repeat_interleave(values(k), _geometric(k, 1.0 / mean_run, gen))])
    return x[:n].contiguous()


def step_function(n, gen):
    return _runs(n, 200.0, lambda k: torch.randint(0, 1 << 20, (k,), generator=gen, device=DEVICE, dtype=torch.int32),
                 gen)


def zipf_codes(n, gen):
    return _choice(n, _zipf_weights(50, 1.2), gen).to(torch.int32)


def normal_with_outliers(n, gen):
    x = torch.round(torch.randn(n, generator=gen, device=DEVICE) * 50.0 + 1000.0).to(torch.int32)
    out = torch.randint(0, 2**31 - 1, (n,), generator=gen, device=DEVICE, dtype=torch.int32)
    return torch.where(torch.rand(n, generator=gen, device=DEVICE) < 0.01, out, x)


def price_walk_f64(n, gen):
    cents = 10_000 + torch.round(torch.randn(n, generator=gen, device=DEVICE)).to(torch.int64).cumsum(0)
    return cents.to(torch.float64) / 100.0


def price_walk_f32(n, gen):
    return price_walk_f64(n, gen).to(torch.float32)


def sensor_levels(n, gen):
    return torch.round(torch.randn(n, generator=gen, device=DEVICE) * 300.0 + 2_000.0).clamp_(0, 4_095).to(torch.int16)


def states(n, gen):
    return _runs(n, 60.0, lambda k: torch.randint(0, 12, (k,), generator=gen, device=DEVICE, dtype=torch.int8), gen)


def mostly_constant(n, gen):
    x = torch.randint(-200, 200, (n,), generator=gen, device=DEVICE, dtype=torch.int16)
    return torch.where(torch.rand(n, generator=gen, device=DEVICE) < 0.03, x, torch.full_like(x, 7))


def volumes(n, gen):
    """Lots of 100, sizes with a Zipf(1.5) tail up to 10^5 distinct values."""
    u = _uniform(n, gen).to(torch.float64)
    return ((torch.floor(u.pow(-2.0)).clamp_(max=1e15).to(torch.int64) % 100_000) * 100).to(torch.int32)


def categories(n, gen):
    return torch.randint(0, 50, (n,), generator=gen, device=DEVICE, dtype=torch.int32)


# (generator, type, tree, bytes of a row in the column, about how many in the blob)
DELTA_AFL = [g.DELTA, g.AFL, g.NONE]
VOLUME_TREE = [g.DICT, g.NONE, g.SCALE, g.DICT, g.NONE, g.AFL, g.NONE]
TABLES = {
    "int": [(timestamps, g.D_INT, DELTA_AFL, 4, 0.75),
            (step_function, g.D_INT, [g.RLE, g.AFL, g.NONE, g.AFL, g.NONE], 4, 0.02),
            (zipf_codes, g.D_INT, [g.DICT, g.NONE, g.NONE], 4, 1.98),
            (normal_with_outliers, g.D_INT, [g.PATCH, g.AFL, g.NONE, g.AFL, g.NONE], 4, 4.0)],
    "float": [(price_walk_f64, g.D_DOUBLE, [g.GFC, g.NONE, g.NONE], 8, 6.4),
              (price_walk_f64, g.D_DOUBLE, [g.FLOAT_TO_INT, g.DELTA, g.AFL, g.NONE], 8, 4.0),
              (price_walk_f32, g.D_FLOAT, [g.GFC, g.NONE, g.NONE], 4, 2.6),
              (price_walk_f32, g.D_FLOAT, [g.FLOAT_TO_INT, g.SCALE, g.DELTA, g.AFL, g.NONE], 4, 4.0)],
    "mixed": [(times_us, g.D_TIME, DELTA_AFL, 8, 1.75),
              (sensor_levels, g.D_SHORT, [g.SCALE, g.AFL, g.NONE], 2, 1.5),
              (states, g.D_CHAR, [g.RLE, g.NONE, g.NONE], 1, 0.08),
              (mostly_constant, g.D_SHORT, [g.CONST, g.NONE], 2, 0.19),
              (volumes, g.D_INT, VOLUME_TREE, 4, 1.35)],
    "batch": [(timestamps, g.D_INT, DELTA_AFL, 4, 0.75),
              (price_walk_f64, g.D_DOUBLE, [g.GFC, g.NONE, g.NONE], 8, 6.4),
              (volumes, g.D_INT, VOLUME_TREE, 4, 1.35),
              (categories, g.D_INT, [g.AFL, g.NONE], 4, 0.75)],
}
# (generator, about how many bytes of a row in the blob of the planner's tree)
BLOCKS = [(timestamps, 0.47), (step_function, 0.02), (zipf_codes, 0.58), (normal_with_outliers, 3.95)]
PART = 0.65  # the same of the optimizer's trees on its parts


def _generator(seed):
    return torch.Generator(DEVICE).manual_seed(1_000 + seed)


def _buffer(x):
    """The library's view of a tensor's memory."""
    return g.DeviceBuffer(context(), x.data_ptr(), x.numel() * x.element_size(), owned=False)


class _Bytes:
    """A library buffer for torch.as_tensor, which keeps it alive."""

    def __init__(self, buf, typestr):
        self.buf = buf
        n = buf.nbytes // int(typestr[2:])
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (buf.dev, False), "version": 2}


TYPESTR = {g.D_INT: "<i4", g.D_TIME: "<i8", g.D_FLOAT: "<f4", g.D_DOUBLE: "<f8", g.D_SHORT: "<i2", g.D_CHAR: "|i1"}


def _tensor(buf, typestr="|u1"):
    return torch.as_tensor(_Bytes(buf, typestr), device=DEVICE)


def _blob(buf, about):
    """All of a blob as two overlapping rows: of 0.7 of its usual size (80 bytes
    of headers with it), or where that does not cover it, of the power of two
    that does."""
    n, row = buf.nbytes, int(0.7 * (about + 80))
    if not row <= n <= 2 * row:
        row = 1 << (n.bit_length() - 1)
    return torch.as_strided(_tensor(buf), (2, row), (n - row, 1))


def _lengths(blobs):
    return torch.tensor([b.nbytes for b in blobs])


def _batch_rows(case, i):
    """Lengths from 4,000 rows to the case's largest, spread over the logarithm."""
    at = (i * 0.6180339887498949) % 1.0
    return int(4_001 * (case["max_rows"] / 4_001) ** at)


def _table_columns(case, gen):
    for make, dtype, path, _, _ in TABLES[case["table"]]:
        yield make(case["rows"], gen), dtype, path


def _blocks(case, seed):
    """Parts of a column of event times whose rate changes half-way, or blocks
    of columns of different kinds."""
    gen = _generator(seed)
    if case["kind"] == "optimizer":
        return [timestamps(case["rows"], gen, 0.3 if i < case["parts"] // 2 else 0.25) for i in range(case["parts"])]
    return [BLOCKS[i % len(BLOCKS)][0](case["rows"], gen) for i in range(case["blocks"])]


# ------------------------------------------------------------------ a state
def prepare(case, seed):
    ctx = context()
    gen = _generator(seed)
    s = {"case": case}
    if case["kind"] == "table":
        cols = list(_table_columns(case, gen))
        s["columns"] = [(g.CompressionTree(ctx, path, dtype), x, _buffer(x), dtype) for x, dtype, path in cols]
        torch.cuda.synchronize()
        if case["dir"] == "decode":
            s["blobs"] = [(tree, tree.Compress(buf), dtype) for tree, _, buf, dtype in s["columns"]]
            del s["columns"], cols
    elif case["kind"] == "batch":
        s["keep"], s["columns"] = [], []
        for i in range(case["columns"]):
            make, dtype, path, _, _ = TABLES["batch"][i % 4]
            x = make(_batch_rows(case, i), gen)
            s["keep"].append(x)
            s["columns"].append((_buffer(x), dtype, path))
        s["config"] = {"workers": 16, "range_rows_log2": 16, "wg_per_cu": 4}
    elif case["kind"] in ("optimizer", "learned"):
        s["keep"] = _blocks(case, seed)
        s["blocks"] = [_buffer(x) for x in s["keep"]]
        if case["kind"] == "learned":
            s["planner"] = g.LearnedPlanner(ctx)
            s["planner"].Load(WEIGHTS)
    else:
        n = case["rows"]
        x, y = timestamps(n, gen), categories(n, gen)
        torch.cuda.synchronize()
        s["tree"] = g.CompressionTree(ctx, DELTA_AFL, g.D_INT)
        s["blob"] = s["tree"].Compress(_buffer(x))
        s["stream"] = ctx.fl_pack(_buffer(y), g.D_INT, 6, n)
        count = min(case["range_rows"], n)
        s["begins"] = _begins(case, seed)
        s["count"] = count
        s["keep"] = torch.randint(0, n, (case["fetch"],), generator=gen, device=DEVICE, dtype=torch.int64)
        s["rows"] = _buffer(s["keep"])
        ctx.sync()
    torch.cuda.synchronize()
    return s


def _begins(case, seed):
    """Where the ranges start: one in each equal part of the column."""
    span = (case["rows"] - min(case["range_rows"], case["rows"])) / case["ranges"]
    r = torch.rand(case["ranges"], generator=torch.Generator().manual_seed(seed)).tolist()
    return [int((i + u) * span) for i, u in enumerate(r)]


def run(s):
    case, ctx = s["case"], context()
    kind = case["kind"]
    if kind == "table":
        if case["dir"] == "decode":
            return [_tensor(tree.Decompress(blob), TYPESTR[dtype]) for tree, blob, dtype in s["blobs"]]
        blobs = [tree.Compress(buf) for tree, _, buf, _ in s["columns"]]
        out = [_blob(b, case["rows"] * col[4]) for b, col in zip(blobs, TABLES[case["table"]])]
        out.append(_lengths(blobs))
        if case["dir"] == "roundtrip":
            out += [_tensor(tree.Decompress(b), TYPESTR[dtype])
                    for (tree, _, _, dtype), b in zip(s["columns"], blobs)]
        return out
    if kind == "batch":
        blobs = g.batch_compress(ctx, s["columns"], config=s["config"])
        return [_blob(b, _batch_rows(case, i) * TABLES["batch"][i % 4][4])
                for i, b in enumerate(blobs)] + [_lengths(blobs)]
    if kind == "optimizer":
        opt = g.CompressionOptimizer(ctx)
        blobs = [opt.CompressData(part, g.D_INT) for part in s["blocks"]]
        path = torch.full((64,), -1)
        path[:len(opt.GetOptimalTree())] = torch.tensor(opt.GetOptimalTree())
        return [_blob(b, case["rows"] * PART) for b in blobs] + [_lengths(blobs), path]
    if kind == "learned":
        blobs = []
        for block in s["blocks"]:
            path, _, _ = s["planner"].Plan(block, g.D_INT)
            blobs.append(g.CompressionTree(ctx, path, g.D_INT).Compress(block))
        return [_blob(b, case["rows"] * BLOCKS[i % len(BLOCKS)][1])
                for i, b in enumerate(blobs)] + [_lengths(blobs)]
    out = [_tensor(s["tree"].DecompressRows(s["blob"], b, s["count"]), "<i4") for b in s["begins"]]
    return out + [_tensor(ctx.fl_fetch(s["stream"], g.D_INT, 6, case["rows"], s["rows"]), "<i4")]


# ----------------------------------------------------------- what is needed
def work(case):
    """Columns read once and blobs written once, or the other way round."""
    kind = case["kind"]
    if kind == "table":
        once = case["rows"] * sum(c[3] + c[4] for c in TABLES[case["table"]])
        return {"bytes": once * (2 if case["dir"] == "roundtrip" else 1), "flops": 0}
    if kind == "batch":
        return {"bytes": sum(_batch_rows(case, i) * (TABLES["batch"][i % 4][3] + TABLES["batch"][i % 4][4])
                             for i in range(case["columns"])), "flops": 0}
    if kind == "optimizer":
        return {"bytes": case["parts"] * case["rows"] * (4 + PART), "flops": 0}
    if kind == "learned":
        return {"bytes": sum(case["rows"] * (4 + BLOCKS[i % len(BLOCKS)][1]) for i in range(case["blocks"])), "flops": 0}
    # a range of a delta column needs the deltas before it (6 bits each); a
    # look-up its index, the word it lies in and its value
    count = min(case["range_rows"], case["rows"])
    before = 0.75 * case["ranges"] * (case["rows"] - count) / 2
    return {"bytes": before + case["ranges"] * count * 4.75 + case["fetch"] * 16, "flops": 0}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """Decoded columns, ranges and look-ups are the rows that went in; the
    blobs' bytes and the chosen trees have no value outside the library."""
    kind = case["kind"]
    if kind == "table" and case["dir"] != "encode":
        cols = [x for x, _, _ in _table_columns(case, _generator(seed))]
        return ([None] * (len(cols) + 1) if case["dir"] == "roundtrip" else []) + cols
    if kind != "access":
        return None
    gen, n = _generator(seed), case["rows"]
    x, y = timestamps(n, gen), categories(n, gen)
    at = torch.randint(0, n, (case["fetch"],), generator=gen, device=DEVICE, dtype=torch.int64)
    count = min(case["range_rows"], n)
    return [x[b:b + count].clone() for b in _begins(case, seed)] + [y[at]]
