"""fp32 searches whose candidates are screened in 16 bits (dsx_screen.hip): the results must be those of the fp32 scores, for operands that
f16 holds badly too (subnormal, above its range, norms of very different size), at the edges of the tables' padding and of both sweeps."""

import numpy as np
import pytest

from test_gpu_kernels import dev
from test_oracle import random_csr

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def everything_screened(dsx):
    """Searches that are small for a test are screened too (by default only where that is expected to be faster)."""
    dsx.dsx_testing_set_screen(1)
    yield
    dsx.dsx_testing_set_screen(0)


def search(pkg, dsx, items, queries, k):
    n, dim = items.shape
    rows = (n + 7) // 8 * 8
    cm = np.full((dim, rows), 1e30, dtype=np.float32)      # pad rows: never looked at
    cm[:, :n] = items.T
    dI, dQ = dev(pkg, cm), dev(pkg, queries)
    scores, idx = pkg.DeviceArray((len(queries), k), np.float32), pkg.DeviceArray((len(queries), k), np.uint32)
    pkg.check(dsx.dsx_knn_search(dI.ptr, rows, rows - n, dim, dQ.ptr, len(queries), k, scores.ptr, idx.ptr, None, 0, None))
    return scores.numpy(), idx.numpy()


def best(full, k):
    """The k best of every row: score descending, then column ascending (NaN last)."""
    part = np.argsort(-full, axis=1, kind="stable")[:, :k]
    return np.take_along_axis(full, part, axis=1), part.astype(np.uint32)


def check_against_float64(got_s, got_i, full, k, unit):
    """Scores right for the columns returned, and no column left out whose score lies above the k-th by more than the roundings."""
    want, _ = best(np.nan_to_num(full, nan=-np.inf), k)
    at = np.take_along_axis(full, got_i.astype(np.int64), axis=1)
    assert np.abs(got_s - at).max() <= unit
    assert np.abs(np.sort(at, axis=1)[:, ::-1] - want).max() <= unit
    assert all(len(set(r)) == k for r in got_i.tolist())


# dim on both sides of a step of 64 and no multiple of 4; more than 256 (the other sweep); the smallest batch and table; a ragged table
@pytest.mark.parametrize("n,queries,dim,k", [(65536, 512, 32, 10), (70003, 520, 36, 64), (66001, 513, 64, 256), (131075, 700, 128, 100),
                                             (80000, 512, 260, 20), (65543, 1030, 100, 1)])
def test_integer_vectors(pkg, dsx, rng, n, queries, dim, k):
    """Every score is exact in fp32 and in f16, whatever the order of the sums; many tie."""
    print("[case] screened knn n=%d queries=%d dim=%d k=%d" % (n, queries, dim, k), flush=True)
    items = rng.integers(-3, 4, size=(n, dim)).astype(np.float32)
    q = rng.integers(-3, 4, size=(queries, dim)).astype(np.float32)
    s, i = search(pkg, dsx, items, q, k)
    assert dsx.dsx_knn_last_search_path() == 1
    rs, ri = best(q @ items.T, k)
    assert np.array_equal(s, rs) and np.array_equal(i, ri)


@pytest.mark.parametrize("form", ["unit", "subnormal", "above the range", "one large item", "nan items", "rising", "huge queries"])
def test_operands_that_f16_holds_badly(pkg, dsx, rng, form):
    n, queries, dim, k = 70001, 516, 48, 50
    print("[case] screened knn %s" % form, flush=True)
    items = rng.standard_normal((n, dim), dtype=np.float32) / np.float32(np.sqrt(dim))
    q = rng.standard_normal((queries, dim), dtype=np.float32)
    if form == "subnormal":
        items *= np.float32(3e-6)
    elif form == "above the range":
        items *= np.float32(3e5)
    elif form == "one large item":
        items[n // 2] *= np.float32(1e4)
    elif form == "nan items":
        items[7::13, 5] = np.nan
    elif form == "rising":
        items = np.sort(items, axis=0)
    elif form == "huge queries":
        q[3] *= np.float32(1e6)
    s, i = search(pkg, dsx, items, q, k)
    full = q.astype(np.float64) @ items.astype(np.float64).T
    # dim products, each rounding at most 2^-24 of |q| |w|: rows are compared in units of |q| max |w|
    norms = np.linalg.norm(items.astype(np.float64), axis=1)
    length = np.linalg.norm(q.astype(np.float64), axis=1)[:, None]
    if form == "one large item":       # (its own scores in units of its own norm, the others in units of theirs)
        at, large = np.take_along_axis(full, i.astype(np.int64), axis=1), i == n // 2
        assert large.sum() > queries // 4 and (np.abs(s - at) / (length * norms[n // 2]))[large].max() <= dim * 2.0 ** -24
        s = np.where(large, at, s)
        norms[n // 2] = 0.0
    scale = length * np.nanmax(norms)
    check_against_float64(s / scale, i, full / scale, k, dim * 2.0 ** -24)
    # what f16 cannot hold, or what would let everything pass, is found before the sweep: block by block straight away
    assert dsx.dsx_knn_last_search_path() == {"unit": 1, "subnormal": 1, "nan items": 1, "rising": 2}.get(form, 0)


# both sides of the line for small searches and of the limit for long items; sums stored and in ranges; a spread that raised bounds pay for most (k
# large, vectors long)
@pytest.mark.parametrize("n,queries,dim,k,longest,path", [(65536, 512, 32, 10, 1, 0), (66001, 513, 120, 10, 1, 1), (70001, 1000, 700, 256, 12, 1),
                                                          (70001, 600, 128, 256, 55, 1), (70001, 600, 128, 256, 90, 0), (140001, 560, 900, 256, 55, 1)])
def test_where_searches_are_screened(pkg, dsx, rng, n, queries, dim, k, longest, path):
    print("[case] screened knn by rule n=%d queries=%d dim=%d k=%d longest=%d" % (n, queries, dim, k, longest), flush=True)
    dsx.dsx_testing_set_screen(0)
    items = rng.standard_normal((n, dim), dtype=np.float32)
    items /= np.linalg.norm(items, axis=1, keepdims=True)
    if longest > 1:
        items *= np.exp(rng.normal(0, 0.3, n)).astype(np.float32)[:, None]
        items[n // 3] *= np.float32(longest) * np.linalg.norm(items, axis=1).mean() / np.linalg.norm(items[n // 3])
    q = rng.standard_normal((queries, dim), dtype=np.float32)
    s, i = search(pkg, dsx, items, q, k)
    assert dsx.dsx_knn_last_search_path() == path and dsx.dsx_knn_last_search_repeated() == 0
    some = np.unique(np.concatenate([[0, queries - 1], rng.integers(0, queries, 40)]))
    full = q[some].astype(np.float64) @ items.astype(np.float64).T
    scale = np.linalg.norm(q[some].astype(np.float64), axis=1)[:, None] * np.linalg.norm(items.astype(np.float64), axis=1).max()
    check_against_float64(s[some] / scale, i[some], full / scale, k, dim * 2.0 ** -24)


@pytest.mark.parametrize("dim", [32, 128, 1024])
def test_components_at_half_the_smallest_subnormal(pkg, dsx, rng, dim):
    """Components a little above 2^-25 round up to 2^-24 in both operands: a screened sum is four times the score, and below any bound
    that leaves out the product of the two roundings.  The best items lie behind the first block."""
    n, queries, k = 66000, 512, 20
    print("[case] screened knn tiny components dim=%d" % dim, flush=True)
    c = rng.uniform(1.05, 1.2, n).astype(np.float32)
    c[60000:60000 + 3 * k] = np.float32(1.0001) + np.arange(3 * k, dtype=np.float32) * np.float32(5e-4)
    items = np.repeat(-c[:, None] * np.float32(2.0 ** -25), dim, axis=1)
    q = np.full((queries, dim), 1.0001 * 2.0 ** -25, dtype=np.float32)
    s, i = search(pkg, dsx, items, q, k)
    full = np.repeat(q[:1].astype(np.float64) @ items.astype(np.float64).T, queries, axis=0)
    unit = dim * (1.0001 * 2.0 ** -25) ** 2
    # every score a sum of dim equal products: dim roundings of 2^-24 of it at most, and neighbours lie 5e-4 apart
    check_against_float64(s / unit, i, full / unit, k, dim * 2.0 ** -24 * 1.2)
    assert (i == 60000 + np.arange(k)).all()


# activations with and without a flat part; columns whose norms span four orders; a bias; a filter; both sides of the padding
@pytest.mark.parametrize("batch,kdim,n,k,act,biased,filtered", [(4096, 32, 16384, 10, 0, True, True), (2200, 60, 17003, 100, 3, True, False),
                                                                (2050, 64, 20000, 256, 2, False, True), (520, 508, 70001, 20, 1, True, True)])
def test_layer(pkg, dsx, rng, batch, kdim, n, k, act, biased, filtered):
    print("[case] screened layer batch=%d kdim=%d n=%d k=%d act=%d" % (batch, kdim, n, k, act), flush=True)
    ldx = (kdim + 3) // 4 * 4
    X = np.maximum(rng.standard_normal((batch, ldx), dtype=np.float32), 0)
    W = rng.standard_normal((kdim, n), dtype=np.float32) * np.float32(1 / np.sqrt(kdim))
    W *= (10.0 ** rng.uniform(-4, 0, n)).astype(np.float32)
    bias = (rng.standard_normal(n) - 3).astype(np.float32) if biased else None
    start = end = fidx = None
    if filtered:
        start, end, fidx = random_csr(rng, batch, n, 300)
    dX, dW, db, ds, de, dx = (dev(pkg, a) for a in (X, W, bias, start, end, fidx))
    keys, vals = pkg.DeviceArray((batch, k), np.float32), pkg.DeviceArray((batch, k), np.uint32)
    pkg.check(dsx.dsx_fc_topk(dX.ptr, ldx, dW.ptr, pkg.ptr(db), batch, kdim, n, act, None, k, keys.ptr, vals.ptr, 0, None, pkg.ptr(ds),
                              pkg.ptr(de), pkg.ptr(dx)))
    z = X[:, :kdim].astype(np.float64) @ W.astype(np.float64) + (bias if biased else 0.0)
    y = {0: lambda v: 1 / (1 + np.exp(-v)), 1: np.tanh, 2: lambda v: np.maximum(v, 0), 3: lambda v: v}[act](z)
    if filtered:
        for b in range(batch):
            y[b, fidx[int(start[b]):int(end[b])]] *= 0.0
    # sums of kdim products and the bias, |x| |w| + |b| below 40 here: kdim roundings of 2^-24 of that at the very most, 1e-6 for the
    # activations' own error; slopes are at most 1
    check_against_float64(keys.numpy(), vals.numpy(), y, k, (kdim + 8) * 40 * 2.0 ** -24 / 8 + 1e-6)


def test_layer_above_the_range_is_recomputed(pkg, dsx, rng):
    """A row that f16 cannot hold: its error has no bound, it is computed from scratch; the others are not."""
    batch, kdim, n, k = 512, 256, 65536, 10
    X = rng.standard_normal((batch, kdim), dtype=np.float32)
    X[17] *= np.float32(1e6)
    W = rng.standard_normal((kdim, n), dtype=np.float32)
    dX, dW = dev(pkg, X), dev(pkg, W)
    keys, vals = pkg.DeviceArray((batch, k), np.float32), pkg.DeviceArray((batch, k), np.uint32)
    dsx.dsx_fc_topk_flagged(1)
    pkg.check(dsx.dsx_fc_topk(dX.ptr, kdim, dW.ptr, None, batch, kdim, n, 3, None, k, keys.ptr, vals.ptr, 0, None, None, None, None))
    y = X.astype(np.float64) @ W.astype(np.float64)
    scale = np.linalg.norm(X.astype(np.float64), axis=1)[:, None] * 25
    check_against_float64(keys.numpy() / scale, vals.numpy(), y / scale, k, kdim * 2.0 ** -24)
    pkg.check(dsx.dsx_sync())
    assert dsx.dsx_fc_topk_flagged(1) == 1


def test_without_room_for_the_copies_of_the_table(pkg, dsx, rng):
    """A workspace, a library scratch or a KnnData without the 16-bit copies: the search runs in fp32."""
    n, queries, dim, k = 70000, 520, 64, 20
    items = rng.integers(-3, 4, size=(n, dim)).astype(np.float32)
    q = rng.integers(-3, 4, size=(queries, dim)).astype(np.float32)
    rs, ri = best(q @ items.T, k)
    full, least = dsx.dsx_knn_workspace_bytes(n, dim, queries, k), dsx.dsx_knn_workspace_bytes_least(n, dim, queries, k)
    assert full > least + n * dim * 4
    dI, dQ = dev(pkg, np.ascontiguousarray(items.T)), dev(pkg, q)
    scores, idx = pkg.DeviceArray((queries, k), np.float32), pkg.DeviceArray((queries, k), np.uint32)
    room = pkg.DeviceArray((full,), np.uint8)

    def run(workspace, size):
        scores.upload(np.zeros((queries, k), np.float32))
        rc = dsx.dsx_knn_search(dI.ptr, n, 0, dim, dQ.ptr, queries, k, scores.ptr, idx.ptr, workspace, size, None)
        if rc == 0:
            assert np.array_equal(scores.numpy(), rs) and np.array_equal(idx.numpy(), ri)
        return rc

    for size, path in ((full, 1), (full - 256, 0), (least, 0)):
        assert run(room.ptr, size) == 0 and dsx.dsx_knn_last_search_path() == path
    assert run(room.ptr, least - 256) == -1
    import amazon_dsstne_amd.host_api as host_api
    lib = host_api.load_host_library()
    dsx.dsx_testing_set_allocation_limit(full - 256)
    try:
        for _ in range(2):
            assert run(None, 0) == 0 and dsx.dsx_knn_last_search_path() == 0
        knn = lib.dsstne_knn_create_typed(queries, k, b"fp32")
        assert knn and lib.dsstne_knn_load(knn, items.ctypes.data, n, dim, None) == 0
        s, i = np.empty((queries, k), np.float32), np.empty((queries, k), np.uint32)
        assert lib.dsstne_knn_search(knn, k, q.ctypes.data, queries, s.ctypes.data, i.ctypes.data) == 0
        lib.dsstne_knn_destroy(knn)
        assert np.array_equal(s, rs) and np.array_equal(i, ri) and dsx.dsx_knn_last_search_path() == 0
    finally:
        dsx.dsx_testing_set_allocation_limit(0)


@pytest.mark.parametrize("act,mask", [(0, -1e9), (0, -np.inf), (3, -1e9), (1, -3e38), (2, -70000.0)])
def test_masked_columns(pkg, dsx, rng, act, mask):
    """Retired items are masked by their biases, new ones pushed: neither makes a row be computed again, and the others' bounds do not
    depend on them.  A few columns (behind the first block) lie above f16's range themselves."""
    batch, kdim, n, k = 1024, 128, 40000, 30
    print("[case] masked columns act=%d mask=%g" % (act, mask), flush=True)
    X = np.maximum(rng.standard_normal((batch, kdim), dtype=np.float32), 0)
    W = rng.standard_normal((kdim, n), dtype=np.float32) * np.float32(0.05)
    bias = (rng.standard_normal(n) * 0.3 - (0.5 if act == 2 else 2)).astype(np.float32)
    bias[rng.random(n) < 0.3] = np.float32(mask)
    bias[[3, 20000, 39999]] = np.float32(-65000.0)
    if act < 2:
        bias[[7, 30000]] = np.float32(1e6)
        W[:, 25000] *= np.float32(1e7)
    dX, dW, db = dev(pkg, X), dev(pkg, W), dev(pkg, bias)
    keys, vals = pkg.DeviceArray((batch, k), np.float32), pkg.DeviceArray((batch, k), np.uint32)
    dsx.dsx_fc_topk_flagged(1)
    pkg.check(dsx.dsx_fc_topk(dX.ptr, kdim, dW.ptr, db.ptr, batch, kdim, n, act, None, k, keys.ptr, vals.ptr, 0, None, None, None, None))
    pkg.check(dsx.dsx_sync())
    assert dsx.dsx_fc_topk_flagged(1) == 0
    with np.errstate(over="ignore"):
        z = X.astype(np.float64) @ W.astype(np.float64) + bias
        y = {0: lambda v: 1 / (1 + np.exp(-v)), 1: np.tanh, 2: lambda v: np.maximum(v, 0), 3: lambda v: v}[act](z)
    # |x| |w| + |b| below 20 for the columns whose scores are not flat: kdim + 8 roundings of 2^-24 of it, 1e-6 for the activations
    check_against_float64(keys.numpy(), vals.numpy(), y, k, (kdim + 8) * 20 * 2.0 ** -24 / 4 + 1e-6)


@pytest.mark.parametrize("n,queries,dim,k,path", [(65536, 512, 32, 10, 0), (150000, 1000, 128, 10, 1), (150000, 512, 64, 256, 0)])
def test_searches_are_screened_where_that_is_faster(pkg, dsx, rng, n, queries, dim, k, path):
    dsx.dsx_testing_set_screen(0)
    items = rng.integers(-3, 4, size=(n, dim)).astype(np.float32)
    q = rng.integers(-3, 4, size=(queries, dim)).astype(np.float32)
    s, i = search(pkg, dsx, items, q, k)
    assert dsx.dsx_knn_last_search_path() == path
    rs, ri = best(q @ items.T, k)
    assert np.array_equal(s, rs) and np.array_equal(i, ri)
