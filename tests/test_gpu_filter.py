"""The filter scan: approximate float16 scores with an error bound decide which pairs are scored
exactly, so every result must be the oracle's (within float32 rounding) whatever the approximation
does, and the exact fallback's bit for bit. Sizes at its edges: rows of one chunk to 4 KB, whole and
partial 256-byte pieces, 128-byte halves and 16-byte chunks, one and several rounds of pieces; one query
to several launches; row counts that end in a partial block; masks that let through everything, some,
and fewer rows than k."""

import time

import numpy as np
import pytest

import oracle
from helpers import assert_topk_equivalent, float_tolerance, normalized

pytestmark = pytest.mark.gpu

INT8_SCALE = np.float32(1.0 / 127.0)


def encode(capi, rows, kind):
    """(stored array, dtype, decoded rows)."""
    if kind == "f32":
        return rows, capi.F32, rows
    if kind == "f16":
        half = oracle.f32_to_f16(rows)
        return half, capi.F16, half.astype(np.float32)
    codes = oracle.quantize_i8(rows, INT8_SCALE)
    return codes, capi.I8, oracle.dequantize_i8(codes, INT8_SCALE)


def run(capi, stored, dtype, queries, k, metric, mask=None, flags=0):
    n, dim = stored.shape
    d_rows, d_queries = capi.DeviceArray.from_host(stored), capi.DeviceArray.from_host(queries)
    d_mask = None if mask is None else capi.DeviceArray.from_host(mask)
    store = capi.store_desc(d_rows, n, dim, dtype, float(INT8_SCALE) if dtype == capi.I8 else 1.0)
    desc = capi.search_desc(store, d_queries, queries.shape[0], k, metric, mask=d_mask, flags=flags)
    return capi.search(desc)


CASES = [
    # kind, n, dim, batch, k, metric (0 cosine, 1 dot, 2 L2), share of rows a mask lets through
    ("f16", 9_001, 64, 9, 10, 2, None),        # half a piece
    ("f16", 9_001, 72, 17, 10, 0, 0.5),        # a chunk past half a piece
    ("f16", 20_011, 100, 1, 10, 0, None),      # rows of 200 bytes, one query
    ("f16", 20_011, 136, 33, 10, 2, None),     # a chunk past a piece
    ("f16", 20_011, 300, 65, 20, 0, 0.3),      # rows of 600 bytes
    ("f16", 20_011, 333, 5, 10, 2, None),      # rows at 2-byte alignment
    ("f16", 9_001, 640, 33, 10, 0, None),      # 5 pieces: two rounds, the last slot empty
    ("f16", 9_001, 768, 130, 100, 1, None),    # three launches of query groups
    ("f16", 9_001, 1000, 16, 10, 2, 0.9),      # 8 pieces, the last one partial
    ("f16", 9_001, 2048, 7, 10, 0, None),      # the widest rows
    ("f32", 9_001, 64, 20, 10, 2, None),       # one piece
    ("f32", 20_011, 100, 40, 10, 0, 0.2),      # 400 bytes
    ("f32", 20_011, 333, 3, 10, 0, None),      # rows at 4-byte alignment
    ("f32", 9_001, 600, 12, 10, 2, None),      # 10 pieces: three rounds of 4, two slots empty
    ("f32", 9_001, 1024, 128, 10, 1, None),    # the widest rows
    ("f32", 20_011, 384, 64, 100, 0, 0.5),
    ("i8", 40_013, 100, 9, 10, 0, None),       # rows at 4-byte alignment
    ("i8", 20_011, 128, 17, 10, 2, None),      # half a piece
    ("i8", 20_011, 384, 128, 10, 1, 0.4),      # a piece and a half
    ("i8", 20_011, 777, 33, 10, 0, None),      # rows at any alignment
    ("i8", 9_001, 1024, 5, 200, 2, None),
    ("f16", 20_011, 768, 9, 50, 0, 0.0),       # (only the rows added below): fewer rows than k
    ("f32", 20_011, 301, 9, 50, 2, 0.0),
    ("f16", 20_011, 768, 9, 10, 0, 1.0),
]


@pytest.mark.parametrize("kind,n,dim,batch,k,metric,share", CASES)
def test_filter_scan(gpu, kind, n, dim, batch, k, metric, share):
    capi = gpu
    stored, dtype, decoded = encode(capi, normalized(n, dim, 300 + dim), kind)
    queries = normalized(batch, dim, 400 + batch)
    mask = None
    if share is not None:
        mask = (np.random.default_rng(dim).random(n) < share).astype(np.uint8)
        mask[[3, n - 1, n // 2]] = 1
    idx, val, flags = run(capi, stored, dtype, queries, k, metric, mask)
    assert not flags.any()
    assert_topk_equivalent(idx, val, oracle.scores_f32(decoded, queries, metric, mask), k,
                           float_tolerance(queries, decoded, metric))
    # and bit for bit what the exact fallback, which sums as the VALU and scalar scans do, computes
    exact = run(capi, stored, dtype, queries, k, metric, mask, capi.SEARCH_FORCE_EXACT_PASS)
    assert np.array_equal(idx, exact[0]) and np.array_equal(val.view(np.uint32), exact[1].view(np.uint32))


@pytest.mark.parametrize("kind,dim,scale", [("f32", 768, 1e6), ("f32", 768, 1e-6), ("f32", 1024, 3e18), ("f16", 768, 1e-5),
                                            ("f16", 1024, 3e4)])
def test_magnitudes(gpu, kind, dim, scale):
    # float32 rows outside float16's range, float16 rows that are mostly subnormal or near the largest
    capi = gpu
    n, batch, k = 9_001, 9, 10
    rows = (normalized(n, dim, 61) * np.float32(scale)).astype(np.float32)
    stored, dtype, decoded = encode(capi, rows, kind)
    queries = normalized(batch, dim, 62)
    idx, val, _ = run(capi, stored, dtype, queries, k, 1)
    assert_topk_equivalent(idx, val, oracle.scores_f32(decoded, queries, 1), k,
                           float_tolerance(queries, decoded, 1) - np.float64(1e-7) * (scale < 1e-3))


@pytest.mark.parametrize("metric", [1, 2])
@pytest.mark.parametrize("sampled", [0, -20])
def test_mixed_magnitudes(gpu, metric, sampled):
    # rows whose scales span forty binary orders: most approximate to zero, and with the sampled rows (the
    # multiples of n / 16) at the bottom the largest overflow float16
    capi = gpu
    n, dim, batch, k = 9_001, 640, 5, 10
    rng = np.random.default_rng(63)
    exponents = rng.integers(-20, 21, (n, 1))
    if sampled:
        exponents[np.arange(16) * (n // 16)] = sampled
    rows = normalized(n, dim, 64) * np.exp2(exponents).astype(np.float32)
    queries = normalized(batch, dim, 65)
    if metric == 2:  # distances on every scale
        queries *= np.exp2(np.array([[-20], [-10], [0], [10], [20]])).astype(np.float32)
    idx, val, _ = run(capi, rows, capi.F32, queries, k, metric)
    assert_topk_equivalent(idx, val, oracle.scores_f32(rows, queries, metric), k, float_tolerance(queries, rows, metric))


# Rows thousands (and, with `scale`, hundreds of thousands) of times longer than the ones the row unit is
# sampled from, which are the multiples of n / 16: their float16 operands overflow or are far from the
# unit, and the approximate scores of an overflowing row say nothing.
def _unsampled(n, rng, count):
    return rng.permutation(np.setdiff1d(np.arange(n), np.arange(16) * (n // 16)))[:count]


@pytest.mark.parametrize("dim", [640, 300, 333])  # whole pieces, a partial chunk half, 4-byte alignment
@pytest.mark.parametrize("lexical", [False, True])
@pytest.mark.parametrize("scale", [1, 200])
def test_outlier_rows_dot(gpu, dim, lexical, scale):
    # every query has 3 rows of length 5000 that score 400, 12 of length 300 that score 300, and ordinary
    # rows (all but those times `scale`); clamped, the longest would score about 100 to 200
    capi = gpu
    n, batch, k = 20_000, 8, 10
    rng = np.random.default_rng(66 + dim)
    rows, queries = normalized(n, dim, 67), normalized(batch, dim, 68)
    places = _unsampled(n, rng, batch * 15).reshape(batch, 15)
    for b in range(batch):
        away = rng.standard_normal((3, dim))
        away -= (away @ queries[b])[:, None] * queries[b]
        away /= np.linalg.norm(away, axis=1, keepdims=True)
        rows[places[b, :3]] = scale * 5000.0 * (0.08 * queries[b] + np.sqrt(1 - 0.08 ** 2) * away)
        rows[places[b, 3:]] = scale * (300.0 - 0.01 * np.arange(12)[:, None]) * queries[b]
    if not lexical:
        idx, val, _ = run(capi, rows, capi.F32, queries, k, 1)
        ref = oracle.scores_f32(rows, queries, 1)
        assert all(set(places[b, :3]) <= set(idx[b]) for b in range(batch))
    else:  # a posting list over a few rows
        docs, terms = np.sort(rng.choice(n, 500, replace=False)).astype(np.int32), np.zeros((batch, 1), np.int32)
        offsets, weights = np.array([0, docs.size], np.int64), rng.random(docs.size).astype(np.float32)
        d = [capi.DeviceArray.from_host(a) for a in (rows, queries, offsets, docs, weights, terms)]
        desc = capi.search_desc(capi.store_desc(d[0], n, dim, capi.F32), d[1], batch, k, 1, lex_offsets=d[2], lex_docs=d[3],
                                lex_weights=d[4], lex_doc_count=n, lex_vocab_size=1, query_terms=d[5], lexical_stride=1,
                                dense_weight=0.5)
        idx, val, _ = capi.search(desc)
        lex = oracle.bm25(offsets, docs, weights, terms[0], n)
        ref = oracle.scores_f32(rows, queries, 1)
        ref = np.stack([oracle.fuse(ref[b], lex, oracle.max_positive(lex), 0.5) for b in range(batch)])
    assert_topk_equivalent(idx, val, ref, k, float_tolerance(queries, rows, 1) + 3e-7)


def test_sums_that_overflow_on_the_way(gpu):
    # a row whose float32 sum becomes infinite and would be zero: it ranks first, as the sum says
    capi = gpu
    n, dim, batch, k = 9_001, 640, 5, 10
    rows = normalized(n, dim, 74) * np.float32(1e37)
    places = 100 + 160 * np.arange(50)
    rows[places] = 0.0
    rows[places, 0] = np.float32(1e38)
    rows[4_321] = 0.0
    rows[4_321, :4] = np.float32(3e38) * np.array([1, 1, -1, -1], np.float32)
    queries = np.ones((batch, dim), np.float32) + np.arange(batch, dtype=np.float32)[:, None]
    idx, val, _ = run(capi, rows, capi.F32, queries, k, 1)
    assert (idx[0] == [4_321, *places[:9]]).all() and np.isinf(val[0, 0])
    exact = run(capi, rows, capi.F32, queries, k, 1, flags=capi.SEARCH_FORCE_EXACT_PASS)
    assert np.array_equal(idx, exact[0]) and np.array_equal(val.view(np.uint32), exact[1].view(np.uint32))


@pytest.mark.parametrize("dim", [640, 300, 333])
@pytest.mark.parametrize("length", [5e3, 1e6])
def test_outlier_rows_l2(gpu, dim, length):
    # twenty long rows, queries near some of them, between them and the rest, and near the rest
    capi = gpu
    n, batch, k = 20_000, 9, 10
    rng = np.random.default_rng(69 + dim)
    rows, queries = normalized(n, dim, 70), normalized(batch, dim, 73)
    places = _unsampled(n, rng, 20)
    rows[places] *= np.float32(length)
    queries[:4] = rows[places[:4]] + np.float32(50.0) * queries[:4]
    queries[4:7] = np.float32(0.5) * rows[places[4:7]] + queries[4:7]
    idx, val, _ = run(capi, rows, capi.F32, queries, k, 2)
    assert np.array_equal(idx[:4, 0], places[:4])
    assert_topk_equivalent(idx, val, oracle.scores_f32(rows, queries, 2), k, float_tolerance(queries, rows, 2))


@pytest.mark.parametrize("kind,dim,metric", [("f16", 768, 0), ("f32", 300, 2), ("i8", 333, 0)])
def test_ties_take_the_lowest_rows(gpu, kind, dim, metric):
    # 40 distinct rows, 500 copies of each: the k best are the lowest copies of the best row
    capi = gpu
    n, batch, k = 20_000, 6, 30
    distinct = normalized(40, dim, 71)
    stored, dtype, decoded = encode(capi, distinct[np.arange(n) % 40], kind)
    queries = normalized(batch, dim, 72)
    idx, val, _ = run(capi, stored, dtype, queries, k, metric)
    best = np.argmax(oracle.scores_f32(decoded[:40], queries, metric), axis=1)
    assert np.array_equal(idx, best[:, None] + 40 * np.arange(k)[None, :])
    assert (val == val[:, :1]).all()


def _seconds(capi, desc):
    """Best of four passes over a workspace that is there."""
    size = capi.search_workspace_bytes(desc)
    workspace = capi.DeviceArray(size, np.uint8)
    idx, val = capi.DeviceArray((desc.batch, desc.k), np.int32), capi.DeviceArray((desc.batch, desc.k), np.float32)
    best = np.inf
    for _ in range(5):
        begin = time.perf_counter()
        capi.search_topk(desc, workspace, size, idx, val)
        capi.synchronize()
        best = min(best, time.perf_counter() - begin)
    return best


def _desc(capi, kind, rows, queries, k, metric, mask=None):
    """(descriptor, decoded rows, queries as the scan sees them) of a search over `rows`."""
    n, dim = rows.shape
    options = dict(mask=None if mask is None else capi.DeviceArray.from_host(mask))
    d_queries = capi.DeviceArray.from_host(queries)
    if kind == "i8row":
        codes, scales = oracle.quantize_rows_i8(rows)
        store = capi.store_desc(capi.DeviceArray.from_host(codes), n, dim, capi.I8, 1.0, capi.DeviceArray.from_host(scales))
        options["int8_mode"] = capi.INT8_PER_VECTOR
        qcodes, qscales = oracle.quantize_rows_i8(queries)
        return (capi.search_desc(store, d_queries, queries.shape[0], k, metric, **options),
                oracle.scores_i8i8(codes, scales, qcodes, qscales, mask))
    stored, dtype, decoded = encode(capi, rows, kind)
    store = capi.store_desc(capi.DeviceArray.from_host(stored), n, dim, dtype, float(INT8_SCALE) if kind == "i8" else 1.0)
    return (capi.search_desc(store, d_queries, queries.shape[0], k, metric, **options),
            oracle.scores_f32(decoded, queries, metric, mask))


# Rows that reach a query's threshold by the thousand: a segment that fills is cut to its best keys, so that
# none overflows, and rows that tie with the threshold are dropped by their numbers.
@pytest.mark.parametrize("kind,n,dim,batch,k,metric,masked", [
    ("f16", 100_003, 768, 9, 10, 0, False),
    ("f16", 60_011, 301, 5, 100, 2, True),
    ("f32", 100_003, 333, 6, 30, 1, False),
    ("i8", 100_003, 384, 17, 10, 0, False),
    ("i8", 50_021, 1024, 5, 200, 2, True),
    ("i8row", 100_003, 640, 20, 40, 0, False),
    ("f16", 60_011, 768, 20, 512, 0, False),  # the widest selections: segments of 1024 keys
])
@pytest.mark.parametrize("equal", [True, False])
def test_crowded_thresholds(gpu, kind, n, dim, batch, k, metric, masked, equal):
    # 40% of the rows are copies of one row, or within the bound's error of it, and half of the queries
    # are near it
    capi = gpu
    rng = np.random.default_rng(75 + dim)
    rows, queries = normalized(n, dim, 76), normalized(batch, dim, 77)
    crowd = np.flatnonzero(rng.random(n) < 0.4)
    noise = np.float32(0.0 if equal else 1e-4 / np.sqrt(dim)) * rng.standard_normal((crowd.size, dim), dtype=np.float32)
    rows[crowd] = rows[crowd[0]] + noise
    queries[:batch // 2] = rows[crowd[0]] + np.float32(0.05) * queries[:batch // 2]
    mask = (rng.random(n) < 0.5).astype(np.uint8) if masked else None
    desc, ref = _desc(capi, kind, rows, queries, k, metric, mask)
    idx, val, flags = capi.search(desc)
    assert not flags.any()
    if equal and kind != "i8row":  # (the oracle's ties are the scan's)
        best = crowd if mask is None else crowd[mask[crowd] != 0]
        assert (idx[:batch // 2] == best[:k]).all()
    if kind == "i8row":
        assert_topk_equivalent(idx, val, ref, k)
    else:
        desc.flags = capi.SEARCH_FORCE_EXACT_PASS
        exact = capi.search(desc)
        assert np.array_equal(idx, exact[0]) and np.array_equal(val.view(np.uint32), exact[1].view(np.uint32))


# Few rows, in the corpus or let through by a mask: a wavefront's tile is then 1, 2, 4, ... rows, so that all
# have some, and a block of the sketch has 16, 8, 4, ... slots.
@pytest.mark.parametrize("kind,dim,batch,metric", [("f16", 768, 9, 0), ("f16", 64, 100, 2), ("f32", 640, 16, 1), ("i8", 301, 40, 0),
                                                   ("i8row", 640, 30, 0)])
@pytest.mark.parametrize("n,allowed", [(1_100, None), (2_049, None), (4_100, None), (33_001, None), (40_009, 3), (40_009, 70),
                                       (40_009, 1_500), (40_009, 2_500), (100_003, 17_000)])
def test_few_rows(gpu, kind, dim, batch, metric, n, allowed):
    capi = gpu
    k = 32
    rows, queries = normalized(n, dim, 86), normalized(batch, dim, 87)
    mask = None
    if allowed is not None:
        mask = np.zeros(n, np.uint8)
        mask[np.random.default_rng(88).choice(n, allowed, replace=False)] = 1
    desc, ref = _desc(capi, kind, rows, queries, k, metric, mask)
    idx, val, flags = capi.search(desc)
    assert not flags.any()
    if kind == "i8row":
        assert_topk_equivalent(idx, val, ref, k)
        return
    assert_topk_equivalent(idx, val, ref, k, float_tolerance(queries, encode(capi, rows, kind)[2], metric))
    desc.flags = capi.SEARCH_FORCE_EXACT_PASS
    exact = capi.search(desc)
    assert np.array_equal(idx, exact[0]) and np.array_equal(val.view(np.uint32), exact[1].view(np.uint32))


@pytest.mark.parametrize("kind,dim,batch,k,n,share", [("f16", 100, 16, 170, 60_000, 0.03), ("i8", 922, 5, 170, 40_000, 0.05)])
def test_masks_that_let_few_rows_through_cost_no_more(gpu, kind, dim, batch, k, n, share):
    # fewer rows than 16 per selected key, of rows that take a wavefront each to score
    capi = gpu
    mask = (np.random.default_rng(89).random(n) < share).astype(np.uint8)
    desc, _ = _desc(capi, kind, normalized(n, dim, 90), normalized(batch, dim, 91), k, 0, mask)
    assert len(capi.search_phase_rows(desc)) == 2  # the filter scan
    filtered = _seconds(capi, desc)
    desc.flags = capi.SEARCH_MATERIALIZE
    assert filtered < 3 * _seconds(capi, desc)


# A query of zeros scores every row 0 and takes the lowest ones: a batch padded with such queries costs
# about what the others do.
@pytest.mark.parametrize("kind,dim,batch,zeros,metric,share", [
    ("f16", 768, 16, 7, 0, None), ("f16", 300, 5, 5, 1, 0.3), ("f32", 333, 6, 1, 0, None), ("f32", 640, 64, 32, 1, 0.02),
    ("i8", 384, 8, 4, 0, None), ("i8row", 768, 16, 8, 0, None), ("i8row", 640, 100, 64, 0, 0.0), ("f16", 768, 9, 3, 2, None),
])
def test_queries_of_zeros(gpu, kind, dim, batch, zeros, metric, share):
    capi = gpu
    n, k = 100_003, 10
    rows, queries = normalized(n, dim, 78), normalized(batch, dim, 79)
    mask = None
    if share is not None:
        mask = (np.random.default_rng(80).random(n) < share).astype(np.uint8)
        mask[[70_000, n - 1]] = 1
    plain, _ = _desc(capi, kind, rows, queries, k, metric, mask)
    queries[::batch // zeros][:zeros] = 0.0
    if kind != "i8row":
        rows[2, 1] = np.nan if kind == "f32" else 0.0  # a row whose score is no zero
    desc, ref = _desc(capi, kind, rows, queries, k, metric, mask)
    idx, val, _ = capi.search(desc)
    if kind == "i8row":
        assert_topk_equivalent(idx, val, ref, k)
    else:
        decoded = encode(capi, rows, kind)[2]
        assert_topk_equivalent(idx, val, ref, k, np.nan_to_num(float_tolerance(queries, decoded, metric)))
    assert _seconds(capi, desc) < 10 * _seconds(capi, plain)


def test_non_finite(gpu):
    # infinite and NaN components follow the float32 sum: +inf ranks first, NaN last; a query with a
    # NaN scores NaN everywhere and takes the lowest rows
    capi = gpu
    n, dim, batch, k = 9_001, 768, 8, 10
    rows = normalized(n, dim, 81)
    rows[17, 3], rows[4_321, 3], rows[900, 5] = np.inf, np.inf, np.nan
    queries = normalized(batch, dim, 82)
    queries[:, 3] = np.abs(queries[:, 3]) + np.float32(0.01)
    queries[2, 9] = np.nan
    queries[3, 3] = -queries[3, 3]
    idx, val, _ = run(capi, rows, capi.F32, queries, k, 0)
    assert np.array_equal(idx[2], np.arange(k)) and np.isnan(val[2]).all()
    assert not np.isin(idx[3], [17, 4_321, 900]).any()
    for q in (0, 1, 4, 7):
        assert idx[q, :2].tolist() == [17, 4_321] and np.isinf(val[q, :2]).all()
    assert not (np.delete(idx, 2, axis=0) == 900).any()


@pytest.mark.parametrize("kind,dim,metric,batch,n,masked", [
    ("f16", 768, 0, 9, 20_011, 0.05),
    ("i8", 333, 1, 17, 20_011, 0.5),
    ("f32", 300, 2, 5, 60_017, 0.0003),  # masked rows sought over several steps, about as many as are selected
    ("f16", 100, 0, 5, 60_017, 0.0),     # a single masked row, the last one
])
def test_masked_rows_outrank_nan_and_minus_infinity(gpu, kind, dim, metric, batch, n, masked):
    # a query for which every allowed row scores NaN (cosine, dot) or -inf (L2): the masked rows, lowest
    # first and wherever they lie, come before those
    capi = gpu
    k = 10
    stored, dtype, decoded = encode(capi, normalized(n, dim, 83), kind)
    queries = normalized(batch, dim, 84)
    bad = batch // 2
    queries[bad, 7] = np.float32(1e30) if metric == 2 else np.nan
    mask = (np.random.default_rng(85).random(n) >= masked).astype(np.uint8)
    mask[:3 * k], mask[n - 1] = 1, 0
    idx, val, _ = run(capi, stored, dtype, queries, k, metric, mask)
    hidden, allowed = np.flatnonzero(mask == 0)[:k], np.flatnonzero(mask)
    assert np.array_equal(idx[bad], np.concatenate([hidden, allowed])[:k])
    assert (val[bad, :hidden.size] == -np.finfo(np.float32).max).all()
    assert not np.isfinite(val[bad, hidden.size:]).any()
    good = np.arange(batch) != bad
    assert_topk_equivalent(idx[good], val[good], oracle.scores_f32(decoded, queries[good], metric, mask), k,
                           float_tolerance(queries[good], decoded, metric))


@pytest.mark.parametrize("kind,dim,metric", [("f16", 768, 0), ("f16", 301, 2), ("i8", 100, 0), ("f32", 333, 1)])
def test_overflowing_segments_fall_back(gpu, kind, dim, metric):
    capi = gpu
    n, batch, k = 40_011, 11, 150
    stored, dtype, decoded = encode(capi, normalized(n, dim, 91), kind)
    queries = normalized(batch, dim, 92)
    mask = np.ones(n, np.uint8)
    mask[::3] = 0
    idx, val, flags = run(capi, stored, dtype, queries, k, metric, mask, capi.SEARCH_TEST_TINY_SEGMENTS)
    assert flags.any()
    plain = run(capi, stored, dtype, queries, k, metric, mask)
    assert np.array_equal(idx, plain[0]) and np.array_equal(val, plain[1])
    assert_topk_equivalent(idx, val, oracle.scores_f32(decoded, queries, metric, mask), k,
                           float_tolerance(queries, decoded, metric))


# per-vector int8 at row widths the int8 matrix-core scan does not take, with masks, and small batches
@pytest.mark.parametrize("n,dim,batch,k,share", [
    (9_001, 16, 6, 10, None),       # one chunk
    (20_011, 272, 33, 10, None),    # a chunk past a piece
    (20_011, 640, 130, 100, 0.5),   # two launches
    (9_001, 1008, 17, 50, 0.0),     # fewer rows than k
    (20_011, 768, 128, 10, 0.3),
    (100_003, 768, 5, 10, None),
])
def test_per_vector_int8_bit_exact(gpu, n, dim, batch, k, share):
    capi = gpu
    codes, scales = oracle.quantize_rows_i8(normalized(n, dim, 500 + dim))
    queries = normalized(batch, dim, 501)
    mask = None
    if share is not None:
        mask = (np.random.default_rng(dim).random(n) < share).astype(np.uint8)
        mask[[3, n - 1]] = 1
    d_codes, d_scales, d_queries = (capi.DeviceArray.from_host(a) for a in (codes, scales, queries))
    d_mask = None if mask is None else capi.DeviceArray.from_host(mask)
    desc = capi.search_desc(capi.store_desc(d_codes, n, dim, capi.I8, 1.0, d_scales), d_queries, batch, k, capi.COSINE,
                            mask=d_mask, int8_mode=capi.INT8_PER_VECTOR)
    idx, val, flags = capi.search(desc)
    qcodes, qscales = oracle.quantize_rows_i8(queries)
    ref_idx, ref_val = oracle.topk(oracle.scores_i8i8(codes, scales, qcodes, qscales, mask), k)
    assert not flags.any()
    assert np.array_equal(idx, ref_idx) and np.array_equal(val, ref_val)


# hybrid searches: the bounds go through the fusion; both ends of the weight
@pytest.mark.parametrize("kind,n,dim,batch,k,metric,weight", [
    ("f16", 20_011, 768, 9, 10, 0, 0.7),
    ("f16", 20_011, 301, 33, 10, 0, 0.3),   # rows of no whole chunks, two launches
    ("f32", 20_011, 100, 20, 50, 2, 0.5),
    ("f32", 9_001, 1024, 16, 10, 1, 0.0),   # only the lexical scores decide (most tie at zero)
    ("f16", 9_001, 100, 5, 10, 0, 1.0),
])
def test_hybrid(gpu, kind, n, dim, batch, k, metric, weight):
    capi = gpu
    stored, dtype, decoded = encode(capi, normalized(n, dim, 600 + dim), kind)
    queries = normalized(batch, dim, 601)
    rng = np.random.default_rng(602)
    vocab, stride = 50, 4
    counts = rng.integers(0, n // 10, vocab)
    docs = np.concatenate([np.sort(rng.choice(n, c, replace=False)) for c in counts]).astype(np.int32)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    weights = rng.random(docs.size).astype(np.float32)
    terms = np.stack([rng.choice(vocab, stride, replace=False) for _ in range(batch)]).astype(np.int32)
    terms[0] = -1  # a query without terms: no lexical part
    d = [capi.DeviceArray.from_host(a) for a in (stored, queries, offsets, docs, weights, terms)]
    desc = capi.search_desc(capi.store_desc(d[0], n, dim, dtype), d[1], batch, k, metric, lex_offsets=d[2], lex_docs=d[3],
                            lex_weights=d[4], lex_doc_count=n, lex_vocab_size=vocab, query_terms=d[5],
                            lexical_stride=stride, dense_weight=weight)
    idx, val, flags = capi.search(desc)
    dense = oracle.scores_f32(decoded, queries, metric)
    fused = np.empty_like(dense)
    for b in range(batch):
        lex = oracle.bm25(offsets, docs, weights, terms[b], n)
        fused[b] = oracle.fuse(dense[b], lex, oracle.max_positive(lex), weight)
    # the dense part's rounding, and that of the fusion's three operations on values of at most 1
    tol = np.float32(weight) * float_tolerance(queries, decoded, metric) + 3e-7
    assert_topk_equivalent(idx, val, fused, k, tol)
    desc.flags = capi.SEARCH_FORCE_EXACT_PASS
    exact = capi.search(desc)
    assert np.array_equal(idx, exact[0]) and np.array_equal(val.view(np.uint32), exact[1].view(np.uint32))


# float32 batches of the matrix-core scan's widths: every 8th tile, then the rest with its exact threshold
def test_two_phases(gpu):
    capi = gpu
    n, dim, batch, k = 400_003, 128, 40, 25
    rows, queries = normalized(n, dim, 95), normalized(batch, dim, 96)
    desc, ref = _desc(capi, "f32", rows, queries, k, 0)
    assert sum(capi.search_phase_rows(desc)) == n
    idx, val, flags = capi.search(desc)
    assert not flags.any()
    assert_topk_equivalent(idx, val, ref, k, float_tolerance(queries, rows, 0))
    for flag in (capi.SEARCH_FORCE_EXACT_PASS, capi.SEARCH_TEST_TINY_SEGMENTS):
        desc.flags = flag
        other = capi.search(desc)
        assert flag == capi.SEARCH_FORCE_EXACT_PASS or other[2].any()
        assert np.array_equal(idx, other[0]) and np.array_equal(val.view(np.uint32), other[1].view(np.uint32))


def test_infinite_scores_rank_as_in_the_split_scan(gpu):
    # 256 and 384 components: launches of 32 to 128 queries rank an infinite score last, as the split scan of
    # smaller corpora does (test_non_finite_rows_depend_on_the_scan); the 22 queries past 128 rank it first
    capi = gpu
    n, dim, batch, k = 400_003, 256, 150, 10
    rows, queries = normalized(n, dim, 97), normalized(batch, dim, 98)
    rows[7, 5] = np.inf
    queries[:, 5] = np.abs(queries[:, 5]) + np.float32(0.01)
    idx, val, _ = run(capi, rows, capi.F32, queries, k, 1)
    assert not (idx[:128] == 7).any() and np.isfinite(val[:128]).all()
    assert (idx[128:, 0] == 7).all() and np.isinf(val[128:, 0]).all()
    rows[7] = 0.0
    finite = run(capi, rows, capi.F32, queries, k, 1)
    assert np.array_equal(idx[:128], finite[0][:128]) and np.array_equal(idx[128:, 1:], finite[0][128:, :-1])
