"""Kernels at the sizes where their work splits can go wrong (edges of tiles,
of workgroups and of the ranges a dispatch rule covers), against NumPy or the
oracle.  Every comparison is exact."""
import math

import numpy as np
import pytest

import gputimeseriescompressionoptimizer_amd as g
from oracle import oracle as O

pytestmark = pytest.mark.gpu

INT_TYPES = [g.D_CHAR, g.D_SHORT, g.D_INT, g.D_TIME]


def _mix64(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _bit_lengths(u):
    return np.array([int(v).bit_length() for v in u])


def _distinct_estimate(x):
    """The 64-register HyperLogLog estimate of the statistics pass."""
    u = np.unique(x)
    u = u.view(f"u{u.itemsize}").astype(np.uint64)
    with np.errstate(over="ignore"):
        h = _mix64(u + np.uint64(0x9E3779B97F4A7C15))
    reg = (h >> np.uint64(58)).astype(np.int64)
    rank = 64 - _bit_lengths((h << np.uint64(6)) | np.uint64(1 << 5)) + 1
    regs = np.zeros(64, np.int64)
    np.maximum.at(regs, reg, rank)
    est = 0.709 * 64 * 64 / sum(math.ldexp(1.0, -int(r)) for r in regs)
    zeros = int((regs == 0).sum())
    if est <= 160 and zeros:
        est = 64.0 * math.log(64.0 / zeros)
    return min(est, float(x.size))


# one workgroup takes 4096 bytes x 4 of rows; 256 and 512 workgroups are the
# fold's own thread count and the largest grid
@pytest.mark.parametrize("dtype", INT_TYPES)
@pytest.mark.parametrize("n", [1, 2, 255, 4096, 4097, 65_537, 2_200_003])
def test_stats_features(ctx, dtype, n):
    npdt = g.NP_DTYPE[dtype]
    r = np.random.default_rng(n)
    info = np.iinfo(npdt)
    x = r.integers(info.min, info.max, n, dtype=npdt, endpoint=True) >> r.integers(0, 8 * npdt().itemsize, n).astype(npdt)
    x[n // 3: n // 2] = 7  # a run: one width, one register
    s = ctx.stats(ctx.upload(x), dtype)
    w = x.astype(np.int64)
    zig = ((w << 1) ^ (w >> 63)).view(np.uint64)
    width = lambda u: np.where(u == 0, 0, np.floor(np.log2(np.maximum(u, 1).astype(np.longdouble))).astype(np.int64) + 1)
    assert list(s.bit_hist) == list(np.bincount(width(zig), minlength=65))
    with np.errstate(over="ignore"):
        d = (x[1:] - x[:-1]).astype(np.int64) if n > 1 else np.zeros(1, np.int64)  # wraps in the type
    assert s.delta_bits_max == (int(width(((d << 1) ^ (d >> 63)).view(np.uint64)).max()) if n > 1 else 0)
    assert s.runs == 1 + int(np.count_nonzero(x[1:] != x[:-1]))
    assert abs(s.distinct_est - _distinct_estimate(x)) <= 0.5 + 1e-9 * s.distinct_est  # rounded to a whole number


def _top(x, k):
    """The k most frequent values, equal counts by the smaller value."""
    v, c = np.unique(x, return_counts=True)
    return [int(v[i]) for i in np.lexsort((v, -c))[:k]]


# 8192 rows a workgroup (4096 of 8 bytes), 64 tables of 4096 slots in the merge;
# 300,000 keys need the global one
@pytest.mark.parametrize("distinct", [1, 3, 4, 63, 2_049, 6_144, 12_289, 45_875, 45_876, 70_000, 300_000])
@pytest.mark.parametrize("dtype", [g.D_INT, g.D_TIME])
def test_most_frequent(ctx, dtype, distinct):
    npdt = g.NP_DTYPE[dtype]
    r = np.random.default_rng(distinct)
    values = r.permutation(np.arange(-(distinct // 2), distinct - distinct // 2, dtype=np.int64) * 1_000_003 + 7)
    x = np.concatenate([values, values[r.integers(0, min(distinct, 40), 20_011)]]).astype(npdt)
    r.shuffle(x)
    meta = g.Encoding(ctx, g.DICT).Encode(ctx.upload(x), dtype)[1].to_bytes()
    want = O.encode(g.DICT, dtype, x)
    assert meta == want[1]
    found = np.frombuffer(meta[16:16 + npdt().itemsize * min(distinct, 4)], npdt)
    assert sorted(int(v) for v in found) == sorted(_top(x, 4))


def test_most_frequent_all_counts_tie(ctx):
    x = np.random.default_rng(1).permutation(np.arange(-50_000, 50_000, dtype=np.int32))
    meta = g.Encoding(ctx, g.DICT).Encode(ctx.upload(x), g.D_INT)[1].to_bytes()
    assert sorted(np.frombuffer(meta[16:32], np.int32)) == [-50_000, -49_999, -49_998, -49_997]


def _hist_ms(ctx, x, dtype):
    """The histogram kernels' time in one dictionary encode, the least of five."""
    buf, enc = ctx.upload(x), g.Encoding(ctx, g.DICT)
    enc.Encode(buf, dtype)
    best = math.inf
    ctx.profile(True)
    for _ in range(5):
        ctx.profile_reset()
        enc.Encode(buf, dtype)
        best = min(best, sum(t[0] for k, t in ctx.kernel_table().items() if k.startswith("k_hist")))
    ctx.profile(False)
    return best


# strides that one multiplication by the golden ratio's bits packs together
@pytest.mark.parametrize("stride", [1, 5_473, 10_946, 50_549, 61_495])
@pytest.mark.parametrize("dtype", [g.D_INT, g.D_TIME])
@pytest.mark.parametrize("distinct,n", [(10_000, 10_000), (2_000, 100_000)])
def test_most_frequent_of_arithmetic_progressions(ctx, dtype, stride, distinct, n):
    """Right, and no slower than random keys: 3 is far above the spread of a
    kernel's time and far below what clustered keys cost (5 to 200)."""
    npdt = g.NP_DTYPE[dtype]
    r = np.random.default_rng(stride)
    at = np.arange(n) if n == distinct else r.integers(0, distinct, n)
    x = (1_400_000_000 + at * stride).astype(npdt)
    assert [o.to_bytes() for o in g.Encoding(ctx, g.DICT).Encode(ctx.upload(x), dtype)] == O.encode(g.DICT, dtype, x)
    other = r.choice(np.iinfo(npdt).max, distinct, replace=False) if dtype == g.D_INT else \
        np.unique(r.integers(0, np.iinfo(npdt).max, distinct + 10))[:distinct]
    assert _hist_ms(ctx, x, dtype) <= 3 * _hist_ms(ctx, r.permutation(other)[at].astype(npdt), dtype)


@pytest.mark.parametrize("n", [10_000, 40_000])
def test_most_frequent_of_keys_with_one_hash(ctx, n):
    """Keys whose folded halves are equal start at one slot with one step; each
    table gives up on them in turn, up to the one that takes every column."""
    hi = np.arange(1, n + 1, dtype=np.uint64)
    lo = (hi * np.uint64(0x85EBCA6B) ^ np.uint64(0x1234567)) & np.uint64(0xFFFFFFFF)
    x = np.random.default_rng(n).permutation(((hi << np.uint64(32)) | lo).astype(np.int64))
    x[::7] = x[3]
    assert [o.to_bytes() for o in g.Encoding(ctx, g.DICT).Encode(ctx.upload(x), g.D_TIME)] == O.encode(g.DICT, g.D_TIME, x)


# 8,192 rows a workgroup (4,096 of 8 bytes) up to 256 of them; past that 16,384
# first, and where its table does not hold the keys, 8,192 in up to 1024 workgroups
@pytest.mark.parametrize("dtype,n,distinct,tables", [
    (g.D_INT, 12_289, 12_289, True), (g.D_INT, 100_000, 16_000, True), (g.D_SHORT, 100_000, 60_000, True),
    (g.D_INT, 256 * 8_192, 30_000, True), (g.D_INT, 256 * 8_192 + 1, 30_000, True),
    (g.D_INT, 1_024 * 8_192, 12_000, True), (g.D_INT, 1_024 * 8_192 + 1, 12_000, False),
    (g.D_TIME, 10_241, 10_241, True), (g.D_DOUBLE, 13_000, 13_000, True), (g.D_FLOAT, 300_000, 30_000, True),
    (g.D_TIME, 256 * 4_096, 30_000, True), (g.D_TIME, 256 * 4_096 + 1, 30_000, True),
    (g.D_DOUBLE, 1_024 * 4_096, 12_000, True), (g.D_TIME, 1_024 * 4_096 + 1, 12_000, False),
])
def test_most_frequent_of_many_keys(ctx, dtype, n, distinct, tables):
    """Columns whose keys the workgroups' tables hold are not counted again in
    the global one (k_hist_init empties that)."""
    npdt = g.NP_DTYPE[dtype]
    r = np.random.default_rng(n)
    if dtype in (g.D_FLOAT, g.D_DOUBLE):
        values = np.unique(r.standard_normal(distinct + 100).astype(npdt))
    else:
        i = np.iinfo(npdt)
        values = np.unique(r.integers(i.min, i.max, 2 * distinct, dtype=npdt)) if dtype != g.D_SHORT else \
            np.arange(-30_000, 30_000).astype(npdt)
    values = r.permutation(values)[:distinct]
    x = r.permutation(np.concatenate([values, values[r.integers(0, values.size, n - values.size)]]))
    x[::113] = values[5]
    x[7::211] = values[6]
    buf, enc = ctx.upload(x), g.Encoding(ctx, g.DICT)
    ctx.profile(True)
    ctx.profile_reset()
    meta = enc.Encode(buf, dtype)[1].to_bytes()
    ran = ctx.kernel_table()
    ctx.profile(False)
    v, c = np.unique(x, return_counts=True)
    want = [v[j] for j in np.lexsort((v, -c))[:4]]
    assert sorted(np.frombuffer(meta[16:16 + 4 * npdt().itemsize], npdt)) == sorted(want)
    assert ("k_hist_init" not in ran) == tables


# past 8M rows (4M of 8 bytes) a first global table of 65,536 slots turns keys
# away, before that the merge's do; the next table holds the column
@pytest.mark.parametrize("dtype,n,distinct,tables", [
    (g.D_INT, 9_000_000, 100_000, 2), (g.D_TIME, 4_200_000, 60_000, 2), (g.D_INT, 400_000, 400_000, 1),
    (g.D_TIME, 2_000_000, 700_000, 1), (g.D_INT, 9_000_000, 40_000, 1), (g.D_INT, 9_000_000, 46_000, 2)])
def test_most_frequent_table_is_sized_by_keys(ctx, dtype, n, distinct, tables):
    """A larger global table has room for a few times the keys, however many
    rows they have."""
    npdt = g.NP_DTYPE[dtype]
    r = np.random.default_rng(n)
    values = r.permutation(np.arange(distinct, dtype=np.int64) * 5_003 - 7).astype(npdt)
    x = r.permutation(np.concatenate([values, values[r.integers(0, distinct, n - distinct)]]))
    x[::1_113], x[7::2_211] = values[5], values[6]
    buf, enc = ctx.upload(x), g.Encoding(ctx, g.DICT)
    ctx.profile(True)
    ctx.profile_reset()
    meta = enc.Encode(buf, dtype)[1].to_bytes()
    _, launches, nbytes = ctx.kernel_table()["k_hist_init"]
    ctx.profile(False)
    assert sorted(np.frombuffer(meta[16:16 + 4 * npdt().itemsize], npdt)) == sorted(_top(x, 4))
    # 16 bytes a slot; twice the keys that the tables before it held and turned
    # away (none of them more than once each), estimated within 20% (six sigma),
    # rounded up to a power of two
    assert launches == tables and nbytes <= 16 * (65_536 + 2 * 2 * 1.2 * 2 * distinct)


# 4096-row tiles; up to 4096 of them are scanned by the counting pass's last
# workgroup (its ticket groups begin past 64, its steps take 1024), more by a
# launch of their own
@pytest.mark.parametrize("tiles", [1, 2, 64, 65, 1_023, 1_024, 1_025, 4_096])
@pytest.mark.parametrize("path,dtype", [
    ([g.PATCH, g.AFL, g.NONE, g.AFL, g.NONE], g.D_SHORT),
    ([g.PATCH, g.NONE, g.NONE], g.D_SHORT),
    ([g.DICT, g.NONE, g.NONE], g.D_CHAR),
    ([g.CONST, g.NONE], g.D_SHORT),
    ([g.RLE, g.NONE, g.NONE], g.D_CHAR),
    ([g.DELTA, g.AFL, g.NONE], g.D_SHORT),
    ([g.DELTA, g.NONE], g.D_SHORT),
], ids=["patch-fl", "patch", "dict", "const", "rle", "delta-fl", "delta"])
def test_tile_scan(ctx, path, dtype, tiles):
    npdt = g.NP_DTYPE[dtype]
    r = np.random.default_rng(tiles)
    for n in (4096 * tiles - 1, 4096 * tiles, 4096 * tiles + 1):  # one tile more with the last
        x = (r.integers(0, 100, n) + (r.random(n) < 0.02) * r.integers(0, 27, n)).astype(npdt)
        x[n // 5: n // 4] = 3
        tree = g.CompressionTree(ctx, path, dtype)
        blob = tree.Compress(ctx.upload(x))
        assert blob.to_bytes() == O.compress(O.tree_from_path(path, dtype), x)
        assert np.array_equal(tree.Decompress(blob).to_numpy(npdt), x)


# scanned with the count (up to 4096 tiles of 4096 rows), whose result says so,
# and by a launch of its own, after which the merge's error flag does
@pytest.mark.parametrize("n,dtype", [(5_000, g.D_INT), (5_000_000, g.D_INT), (4_096 * 4_096, g.D_SHORT),
                                     (4_096 * 4_096 + 1, g.D_SHORT)])
def test_merge_outputs_too_short(ctx, n, dtype):
    """A stencil with more set or clear bits than the outputs hold is refused."""
    npdt = g.NP_DTYPE[dtype]
    x = (np.arange(n) % 5).astype(npdt)
    enc = g.Encoding(ctx, g.DICT)
    stencil, codes, rest = enc.Encode(ctx.upload(x), dtype)
    flipped = ctx.upload(np.bitwise_xor(np.frombuffer(stencil.to_bytes(), np.uint8),
                                        np.r_[np.zeros(1, np.uint8), np.full(stencil.nbytes - 1, 255, np.uint8)]))
    with pytest.raises(g.DdjError) as e:
        enc.Decode([flipped, codes, rest], dtype)
    assert e.value.status == 3
    assert np.array_equal(enc.Decode([stencil, codes, rest], dtype).to_numpy(npdt), x)


@pytest.mark.parametrize("n", [5_000, 1_000_001, 4_096 * 4_096 + 1])
@pytest.mark.parametrize("flip", [0xFF, 0x55])
def test_patch_streams_too_short(ctx, n, flip):
    """The same for a patch whose two sides are FL streams: most tiles ask for
    rows far past the end of one, which are not read."""
    r = np.random.default_rng(n)
    x = np.where(r.random(n) < 0.01, r.integers(20_000, 30_000, n), 500 + np.arange(n) % 90).astype(np.int16)
    path = [g.PATCH, g.AFL, g.NONE, g.AFL, g.NONE]
    tree = g.CompressionTree(ctx, path, g.D_SHORT)
    blob = np.frombuffer(tree.Compress(ctx.upload(x)).to_bytes(), np.uint8)
    stencil = slice(8 + 1, 8 + int(blob[4:8].view(np.int32)[0]))  # after the node's header and the padding's count
    bad = blob.copy()
    bad[stencil] ^= flip
    with pytest.raises(g.DdjError) as e:
        tree.Decompress(ctx.upload(bad))
    assert e.value.status == 3
    assert np.array_equal(tree.Decompress(ctx.upload(blob)).to_numpy(np.int16), x)


@pytest.mark.parametrize("begin,count", [(0, 1), (0, 4097), (1, 1), (4095, 2), (4096, 4096), (4097, 1), (99_999, 1),
                                         (70_001, 29_999), (0, 100_000)])
def test_delta_row_ranges(ctx, begin, count):
    x = np.cumsum(np.random.default_rng(3).integers(0, 60, 100_000)).astype(np.int32)
    tree = g.CompressionTree(ctx, [g.DELTA, g.AFL, g.NONE], g.D_INT)
    blob = tree.Compress(ctx.upload(x))
    assert np.array_equal(tree.DecompressRows(blob, begin, count).to_numpy(np.int32), x[begin:begin + count])


def test_parse_deep_and_wide_blobs(ctx):
    """Node tables up to and past the 64 nodes that come back at once."""
    x = np.random.default_rng(8).integers(0, 1000, 5_000).astype(np.int32)
    for depth in (1, 5, 20, 31, 32, 33, 50):
        path = [g.SCALE] * depth + [g.PATCH, g.DELTA, g.AFL, g.NONE, g.NONE]
        blob = g.CompressionTree(ctx, path, g.D_INT).Compress(ctx.upload(x))
        assert blob.to_bytes() == O.compress(O.tree_from_path(path, g.D_INT), x)
        assert np.array_equal(g.CompressionTree(ctx).Decompress(blob).to_numpy(np.int32), x)
    def both(d):
        return [g.PATCH] + both(d - 1) + both(d - 1) if d else [g.NONE]
    path = both(6)  # 127 nodes
    blob = g.CompressionTree(ctx, path, g.D_INT).Compress(ctx.upload(x))
    assert blob.to_bytes() == O.compress(O.tree_from_path(path, g.D_INT), x)
    assert np.array_equal(g.CompressionTree(ctx).Decompress(blob).to_numpy(np.int32), x)


@pytest.mark.parametrize("rows", [1, 31, 32, 33, 100])
def test_planner_rows_predicted_alone_or_together(ctx, rows):
    """Up to 32 rows go straight to the host, more through device buffers;
    a row's prediction does not depend on the rows beside it."""
    net = g.LearnedPlanner(ctx, seed=5)
    x = np.random.default_rng(rows).standard_normal((rows, g.MLP_FEATURES)).astype(np.float32)
    y = net.Predict(x)
    for i in {0, rows // 2, rows - 1}:
        assert np.array_equal(net.Predict(x[i:i + 1])[0], y[i])


# 12,288 rows (10,240 of 8 bytes) are the most that one workgroup counts; past
# them integer keys within 512 of the first row's are counted by their offset
@pytest.mark.parametrize("dtype", INT_TYPES + [g.D_FLOAT, g.D_DOUBLE])
@pytest.mark.parametrize("n", [1, 5, 10_239, 10_240, 10_241, 12_287, 12_288, 12_289, 40_003])
def test_most_frequent_small_columns_and_windows(ctx, dtype, n):
    npdt = g.NP_DTYPE[dtype]
    r = np.random.default_rng(n)
    if dtype in (g.D_FLOAT, g.D_DOUBLE):
        x = r.integers(-4, 4, n).astype(npdt) * npdt(-0.25)  # zeros of both signs
        x[r.random(n) < 0.01] = np.nan
        every = (r.standard_normal(n) * 1e3).astype(npdt)
    else:
        i = np.iinfo(npdt)
        lo = r.choice([i.min, -1, i.max - 3])  # around the wrap and the all-ones pattern
        x = (lo + (r.integers(0, 1_200, n) * (r.random(n) < 0.4))).astype(npdt)
        every = r.permutation(np.arange(n)).astype(npdt)
    for col in (x, every, np.full(n, x[0], npdt)):
        outs = [o.to_bytes() for o in g.Encoding(ctx, g.DICT).Encode(ctx.upload(col), dtype)]
        assert outs == O.encode(g.DICT, dtype, col)
        outs = [o.to_bytes() for o in g.Encoding(ctx, g.CONST).Encode(ctx.upload(col), dtype)]
        assert outs == O.encode(g.CONST, dtype, col)


@pytest.mark.parametrize("dtype,edge", [(g.D_INT, 512), (g.D_SHORT, 512), (g.D_TIME, 512)])
def test_most_frequent_at_the_window_edges(ctx, dtype, edge):
    npdt = g.NP_DTYPE[dtype]
    for base in (0, np.iinfo(npdt).max, np.iinfo(npdt).min):
        with np.errstate(over="ignore"):
            keys = np.array([base], npdt) + np.array([0, -edge - 1, -edge, -edge + 1, edge - 1, edge, edge + 1], npdt)
        x = np.repeat(keys, [1, 9_001, 9_002, 9_003, 9_004, 9_005, 9_006]).astype(npdt)
        x[1:] = np.random.default_rng(2).permutation(x[1:])
        outs = [o.to_bytes() for o in g.Encoding(ctx, g.DICT).Encode(ctx.upload(x), dtype)]
        assert outs == O.encode(g.DICT, dtype, x)


@pytest.mark.parametrize("dtype,per_tile", [(g.D_INT, 5_000), (g.D_TIME, 2_500)])
@pytest.mark.parametrize("tiles", [40, 257])
def test_most_frequent_many_keys_in_few_rows(ctx, dtype, per_tile, tiles):
    """Every 16384-row tile has keys of its own: they fit the workgroups' tables,
    and with 257 tiles (the last one a second tile of the first workgroup)
    not the partitions' sums."""
    npdt = g.NP_DTYPE[dtype]
    row = np.arange(tiles * 16_384)
    x = ((row // 16_384) * per_tile + row % per_tile).astype(npdt) * npdt(1_003)
    x[::97] = -5
    x[1::1_009] = 77
    meta = g.Encoding(ctx, g.DICT).Encode(ctx.upload(x), dtype)[1].to_bytes()
    assert sorted(np.frombuffer(meta[16:16 + 4 * npdt().itemsize], npdt)) == sorted(_top(x, 4))


@pytest.mark.parametrize("dtype", [g.D_FLOAT, g.D_DOUBLE])
@pytest.mark.parametrize("path", [
    [g.FLOAT_TO_INT, g.DELTA, g.AFL, g.NONE],
    [g.FLOAT_TO_INT, g.SCALE, g.DELTA, g.AFL, g.NONE],
    [g.FLOAT_TO_INT, g.SCALE, g.SCALE, g.DELTA, g.AFL, g.NONE],
    [g.FLOAT_TO_INT, g.FLOAT_TO_INT, g.DELTA, g.AFL, g.NONE],
], ids=["f2i-delta", "f2i-scale-delta", "f2i-scale-scale-delta", "f2i-f2i-delta"])
@pytest.mark.parametrize("n", [1, 2, 3, 4_096, 4_097, 4_098, 8_193, 20_001])
def test_float_rows_written_by_the_delta_decode(ctx, dtype, path, n):
    npdt = g.NP_DTYPE[dtype]
    r = np.random.default_rng(n)
    for scale, step in ((1.0, 1), (4.0, 1), (100.0, 40), (0.0, 0)):  # 0, 2 and 2-3 decimals; not decimal at all
        if scale:
            x = (np.cumsum(r.integers(-step if step > 1 else 0, step + 1, n)) / scale - 5.0).astype(npdt)
        else:
            x = r.standard_normal(n).astype(npdt)
        tree = g.CompressionTree(ctx, path, dtype)
        blob = tree.Compress(ctx.upload(x)).to_bytes()
        assert blob == O.compress(O.tree_from_path(path, dtype), x)
        want = O.decompress(blob)
        for shift in (0, 1, 2, 3):  # the 32-bit deltas at any byte address
            moved = ctx.upload(b"\0" * shift + blob)
            assert tree.Decompress(moved.view(shift, len(blob))).to_bytes() == want, (scale, shift)


@pytest.mark.parametrize("dtype", [g.D_INT, g.D_TIME, g.D_SHORT, g.D_CHAR])
@pytest.mark.parametrize("n", [1, 2, 4_097, 12_290])
def test_scaled_deltas(ctx, dtype, n):
    """scale over delta over FL at the full width (wrapping steps) and a narrow one."""
    npdt = g.NP_DTYPE[dtype]
    r = np.random.default_rng(n)
    i = np.iinfo(npdt)
    path = [g.SCALE, g.DELTA, g.AFL, g.NONE]
    for x in (r.integers(i.min, i.max, n, dtype=npdt, endpoint=True), (50 + np.arange(n) % 60).astype(npdt)):
        tree = g.CompressionTree(ctx, path, dtype)
        blob = tree.Compress(ctx.upload(x)).to_bytes()
        assert blob == O.compress(O.tree_from_path(path, dtype), x)
        for shift in (0, 1, 3):
            moved = ctx.upload(b"\0" * shift + blob)
            assert np.array_equal(tree.Decompress(moved.view(shift, len(blob))).to_numpy(npdt), x)


@pytest.mark.parametrize("dtype", [g.D_FLOAT, g.D_DOUBLE])
@pytest.mark.parametrize("n", [1, 63, 5_000, 300_001])
def test_precision_of_late_rows(ctx, dtype, n):
    """Rows whose decimals grow along the column, one row deciding."""
    npdt = g.NP_DTYPE[dtype]
    x = np.full(n, 2.0, npdt)
    for decimals in (0, 1, 2, 3, 4):
        x[n - 1 - n // 7] = npdt(1.0) + npdt(3) / npdt(10.0 ** decimals)
        outs = [o.to_bytes() for o in g.Encoding(ctx, g.FLOAT_TO_INT).Encode(ctx.upload(x), dtype)]
        assert outs == O.encode(g.FLOAT_TO_INT, dtype, x)
        assert ctx.stats(ctx.upload(x), dtype).precision == O.stats(dtype, x).precision
    x[n // 2] = np.nan
    outs = [o.to_bytes() for o in g.Encoding(ctx, g.FLOAT_TO_INT).Encode(ctx.upload(x), dtype)]
    assert outs == O.encode(g.FLOAT_TO_INT, dtype, x)


# 4096 rows a tile: runs that start, end and stretch at and over the tiles'
# edges, tiles without a run's start, and more tiles than a tail folds (4096)
@pytest.mark.parametrize("dtype", INT_TYPES + [g.D_FLOAT, g.D_DOUBLE])
@pytest.mark.parametrize("n", [1, 4_096, 4_097, 40_961, 2_000_001, 4_096 * 4_097 + 5])
def test_runs_over_tiles(ctx, dtype, n):
    npdt = g.NP_DTYPE[dtype]
    starts = {0, 4_095, 4_096, 8_193, 12_288, 12_289, 32_768, 40_960, 1_048_576, 4_096 * 4_096, n - 1}
    starts |= set(range(49_152, 53_248, 3))  # one tile of short runs
    starts = np.array(sorted(s for s in starts if 0 <= s < n))
    keys = (np.arange(starts.size) * 37 % 101 - 50).astype(npdt)
    x = np.repeat(keys, np.diff(np.append(starts, n)))
    path = [g.RLE, g.AFL, g.NONE, g.AFL, g.NONE] if dtype in INT_TYPES else [g.RLE, g.AFL, g.NONE, g.NONE]
    tree = g.CompressionTree(ctx, path, dtype)
    blob = tree.Compress(ctx.upload(x))
    assert blob.to_bytes() == O.compress(O.tree_from_path(path, dtype), x)
    assert np.array_equal(tree.Decompress(blob).to_numpy(npdt), x)
