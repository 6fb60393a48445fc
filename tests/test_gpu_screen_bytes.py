"""Searches and output layers screened in bytes: the results are those of the searches screened in halves, bit for bit, since either
only decides what is scored in fp32; whole numbers also against a full sort."""

import ctypes as C

import numpy as np
import pytest

from test_gpu_kept_tables import best
from test_gpu_kernels import dev
from test_oracle import random_csr

pytestmark = pytest.mark.gpu

LINEAR, SIGMOID = 3, 0


@pytest.fixture(autouse=True)
def default_switches(pkg, dsx):
    yield
    pkg.check(dsx.dsx_testing_reset())


def layer(pkg, dsx, X, W, bias, act, k, csr=None, mode=1):
    """Keys and values of a layer with a kept table, and whether rows were computed again."""
    batch, kdim, n = X.shape[0], X.shape[1], W.shape[1]
    pkg.check(dsx.dsx_testing_set_screen_bytes(mode))
    dX, dW = dev(pkg, X), dev(pkg, W)
    db = dev(pkg, bias) if bias is not None else None
    ds, de, dx = (dev(pkg, a) for a in csr) if csr else (None, None, None)
    table = pkg.DeviceArray((dsx.dsx_screen_table_bytes(n, kdim),), np.uint8)
    keys, vals = pkg.DeviceArray((batch, k), np.float32), pkg.DeviceArray((batch, k), np.uint32)
    pkg.check(dsx.dsx_screen_table_build(dW.ptr, n, n, kdim, table.ptr))
    dsx.dsx_fc_topk_flagged_for(dW.ptr, 1)
    pkg.check(dsx.dsx_fc_topk_screened(dX.ptr, kdim, dW.ptr, table.ptr, pkg.ptr(db), batch, kdim, n, act, None, k, keys.ptr, vals.ptr, 0, None,
                                       pkg.ptr(ds), pkg.ptr(de), pkg.ptr(dx)))
    got = keys.numpy(), vals.numpy()
    return got[0], got[1], dsx.dsx_fc_topk_flagged_for(dW.ptr, 1)


def search(pkg, dsx, items, q, k, mode=1):
    n, dim = items.shape
    rows = (n + 7) // 8 * 8
    pkg.check(dsx.dsx_testing_set_screen_bytes(mode))
    cm = np.full((dim, rows), 1e30, dtype=np.float32)      # pad rows: never looked at
    cm[:, :n] = items.T
    dI, dQ = dev(pkg, cm), dev(pkg, q)
    room = pkg.DeviceArray((dsx.dsx_knn_workspace_bytes_prepared(rows, dim, len(q), k),), np.uint8)
    prepared = C.c_int(-1)
    pkg.check(dsx.dsx_knn_prepare(dI.ptr, rows, rows - n, dim, len(q), k, room.ptr, room.nbytes, C.byref(prepared)))
    assert prepared.value in (3, 4)
    scores, idx = pkg.DeviceArray((len(q), k), np.float32), pkg.DeviceArray((len(q), k), np.uint32)
    pkg.check(dsx.dsx_knn_search_host(prepared.value, dI.ptr, rows, rows - n, dim, dQ.ptr, len(q), k, scores.ptr, idx.ptr, None, None, room.ptr,
                                      room.nbytes, None))
    return scores.numpy(), idx.numpy(), dsx.dsx_knn_last_search_repeated()


# tile shapes (up to 64, 128 and more rows; few and many tiles), each number of words per lane at both ends, one to nine stages a tile, k at both ends
@pytest.mark.parametrize("batch,kdim,n,k,filtered", [(1, 32, 8192, 1, False), (48, 100, 27278, 20, True), (64, 128, 65536, 33, True),
                                                     (65, 64, 65537, 256, True), (128, 260, 8200, 32, True), (129, 1100, 27278, 100, True),
                                                     (513, 96, 131073, 10, True), (300, 64, 262144, 50, True), (769, 32, 32769, 256, False),
                                                     (3, 36, 1048576, 40, True), (257, 16, 262145, 7, True)])
def test_layer_of_whole_numbers(pkg, dsx, rng, batch, kdim, n, k, filtered):
    print("[case] layer in bytes batch=%d kdim=%d n=%d k=%d" % (batch, kdim, n, k), flush=True)
    X = rng.integers(-3, 4, size=(batch, kdim)).astype(np.float32)
    W = rng.integers(-3, 4, size=(kdim, n)).astype(np.float32)
    bias = rng.integers(-40, 41, size=n).astype(np.float32)
    csr = None
    if filtered:
        start, end, fidx = random_csr(rng, batch, n, 300)
        all_but = np.delete(np.arange(n, dtype=np.uint32), np.arange(0, n, 23))   # of the last row: one column in 23 is left
        fidx = np.concatenate([fidx[:int(start[batch - 1])], all_but]).astype(fidx.dtype)
        end[batch - 1] = len(fidx)
        csr = start, end, fidx
    keys, vals, _ = layer(pkg, dsx, X, W, bias, LINEAR, k, csr)
    y = X @ W + bias
    if filtered:
        for b in range(batch):
            y[b, fidx[int(start[b]):int(end[b])]] = 0
    want_keys, want_vals = best(y, k)
    assert np.array_equal(keys, want_keys)
    # (a zero of a listed column and one of another column tie; which of them is listed first is the path's own)
    assert not (vals != want_vals)[want_keys != 0].any()


@pytest.mark.parametrize("n,dim,queries,k", [(8192, 16, 70, 128), (65601, 768, 520, 100), (400003, 128, 4, 10), (270001, 187, 513, 33), (1048575, 24, 300, 5)])
def test_search_of_whole_numbers(pkg, dsx, rng, n, dim, queries, k):
    print("[case] search in bytes n=%d dim=%d queries=%d k=%d" % (n, dim, queries, k), flush=True)
    items = rng.integers(-3, 4, size=(n, dim)).astype(np.float32)
    q = rng.integers(-3, 4, size=(queries, dim)).astype(np.float32)
    scores, idx, _ = search(pkg, dsx, items, q, k)
    rs, ri = best(q @ items.T, k)
    assert np.array_equal(scores, rs) and np.array_equal(idx, ri)


@pytest.mark.parametrize("form", ["normal", "lognormal", "one long", "tiny", "constant", "sparse", "clusters", "one in two blocks", "one place", "zero and NaN queries", "NaN items"])
def test_search_of_floats(pkg, dsx, rng, form):
    n, dim, queries, k = 270001 if form == "one in two blocks" else 70001, 130, 300, 50
    print("[case] search in bytes, %s" % form, flush=True)
    items = rng.normal(size=(n, dim)).astype(np.float32)
    q = rng.normal(size=(queries, dim)).astype(np.float32)
    if form == "lognormal": items *= rng.lognormal(0, 0.5, size=(n, 1)).astype(np.float32)
    elif form == "one long": items[12345] *= 40
    elif form == "tiny": items *= np.float32(1e-13); q *= np.float32(1e-13)   # (sums of 1e-30 and less are held to be equal)
    elif form == "constant": items = np.sign(items) * np.float32(0.7)   # every component as large as the largest
    elif form == "sparse": items[rng.random(items.shape) < 0.95] = 0
    elif form == "clusters": items = items[rng.integers(0, 400, n)] + items * np.float32(0.01)   # some 175 near each neighbour
    elif form in ("one in two blocks", "one place"):   # as many within the error of the best that lists of words overflow, or several rounds of whole blocks
        near = slice(0, n, 64) if form == "one in two blocks" else slice(100, 6100)
        items[near] = 2 * items[0] + items[near] * np.float32(0.01)
        q = items[0] / 2 + q * np.float32(0.1)
    elif form == "zero and NaN queries": q[7] = 0; q[9, 3] = np.nan
    elif form == "NaN items": items[77, 5] = np.nan; items[78] = np.nan
    got, want = search(pkg, dsx, items, q, k), search(pkg, dsx, items, q, k, mode=2)
    rows = ~np.isnan(q).any(axis=1) & (q != 0).any(axis=1)   # (equal scores of the others: in any order that is the path's own)
    if want[2]:   # (in halves the search was done again in fp32, whose sums have another order: both within dim roundings of the exact sum)
        length = np.sqrt((q[rows].astype(np.float64) ** 2).sum(axis=1)).max() * np.sqrt((items.astype(np.float64) ** 2).sum(axis=1)).max()
        assert np.abs(got[0].astype(np.float64) - want[0])[rows].max() <= 2 * dim * 2.0 ** -24 * length
    else:
        assert np.array_equal(got[0][rows], want[0][rows]) and np.array_equal(got[1][rows], want[1][rows])
    if form != "zero and NaN queries": assert got[2] == 0


@pytest.mark.parametrize("form", ["plain", "masked", "always passes", "own items best", "rising", "zero rows", "small rows", "tied blocks"])
@pytest.mark.parametrize("act", [SIGMOID, LINEAR])
def test_layer_of_floats(pkg, dsx, rng, form, act):
    batch, kdim, n, k = 300, 96, 40000, 30
    print("[case] layer in bytes, %s, activation %d" % (form, act), flush=True)
    X = np.maximum(rng.normal(size=(batch, kdim)), 0).astype(np.float32)
    W = (rng.normal(size=(kdim, n)) / np.sqrt(kdim)).astype(np.float32)
    bias = rng.normal(-1, 0.7, size=n).astype(np.float32)
    start, end, fidx = random_csr(rng, batch, n, 144)
    if form == "masked": bias[::3] = -np.inf; bias[1::3] = np.float32(-1e9)
    elif form == "always passes": W[:, 100] *= np.float32(4e5); W[:, 30000] *= np.float32(-4e5)
    elif form == "own items best":
        top = np.argsort(-(X @ W + bias), axis=1)[:, :200].astype(fidx.dtype)
        fidx = np.sort(top, axis=1).reshape(-1)
        start, end = (np.arange(batch) * 200).astype(start.dtype), ((np.arange(batch) + 1) * 200).astype(end.dtype)
    elif form == "rising": bias = np.linspace(-3, 0, n).astype(np.float32)
    elif form == "zero rows": X[::5] = 0
    elif form == "small rows": X[::5] *= np.float32(1e-3); X[1::5] *= np.float32(1e-6)
    elif form == "tied blocks": W[:, 1::2] = W[:, ::2]; bias[1::2] = bias[::2]   # the second largest of a block is the largest
    csr = start, end, fidx
    got, want = layer(pkg, dsx, X, W, bias, act, k, csr), layer(pkg, dsx, X, W, bias, act, k, csr, mode=2)
    if want[2]:   # (rows computed again in fp32: as above, an activation's slope is 1 at most)
        length = np.sqrt((X.astype(np.float64) ** 2).sum(axis=1)).max() * np.sqrt((W.astype(np.float64) ** 2).sum(axis=0))
        bound = 2 * (kdim + 4) * 2.0 ** -24 * (length + np.abs(np.where(np.isfinite(bias), bias, 0)))
        assert (np.abs(got[0].astype(np.float64) - want[0]) <= np.maximum(bound[got[1]], bound[want[1]])).all()
    else:
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    if act == SIGMOID: assert got[2] == 0


def search_halves(pkg, dsx, items, q, k, storage=None):
    """fp16 storage with the table's bytes kept (storage: another one of the same workspace); scores, indexes, whether it was repeated."""
    n, dim = items.shape
    rows = (n + 7) // 8 * 8
    pkg.check(dsx.dsx_testing_set_screen_bytes(1))
    cm = np.full((dim, rows), 6e4, dtype=np.float32)      # pad rows: never looked at
    cm[:, :n] = items.T
    dI, dQ = dev(pkg, cm), dev(pkg, q)
    table = pkg.DeviceArray((dsx.dsx_knn_f16_table_bytes(rows, dim),), np.uint8)
    pkg.check(dsx.dsx_knn_f16_convert_items(dI.ptr, rows, rows - n, dim, table.ptr))
    room = pkg.DeviceArray((dsx.dsx_knn_workspace_bytes_f16_prepared(rows, dim, len(q), k),), np.uint8)
    prepared = C.c_int(-1)
    pkg.check(dsx.dsx_knn_prepare_f16(table.ptr, rows, rows - n, dim, len(q), k, room.ptr, room.nbytes, C.byref(prepared)))
    if prepared.value == 0: return None
    assert prepared.value == 6
    scores, idx = pkg.DeviceArray((len(q), k), np.float32), pkg.DeviceArray((len(q), k), np.uint32)
    pkg.check(dsx.dsx_knn_search_host(storage or prepared.value, table.ptr, rows, rows - n, dim, dQ.ptr, len(q), k, scores.ptr, idx.ptr, None, None, room.ptr,
                                      room.nbytes, None))
    return scores.numpy(), idx.numpy(), dsx.dsx_knn_last_search_repeated()


@pytest.mark.parametrize("n,dim,queries,k", [(8192, 16, 70, 128), (65601, 768, 520, 100), (400003, 128, 4, 10), (270001, 187, 513, 33), (30001, 300, 300, 256)])
def test_search_of_whole_halves(pkg, dsx, rng, n, dim, queries, k):
    print("[case] halves in bytes n=%d dim=%d queries=%d k=%d" % (n, dim, queries, k), flush=True)
    items = rng.integers(-3, 4, size=(n, dim)).astype(np.float32)
    q = rng.integers(-3, 4, size=(queries, dim)).astype(np.float32)
    rs, ri = best(q @ items.T, k)
    for storage in (6, 7):
        scores, idx, _ = search_halves(pkg, dsx, items, q, k, storage)
        assert np.array_equal(scores, rs) and np.array_equal(idx, ri)


@pytest.mark.parametrize("form", ["normal", "lognormal", "one long", "constant", "infinite items", "infinite query", "tied"])
def test_search_of_halves(pkg, dsx, rng, form):
    n, dim, queries, k = 70001, 130, 300, 50
    print("[case] halves in bytes, %s" % form, flush=True)
    items = rng.normal(size=(n, dim)).astype(np.float32)
    q = rng.normal(size=(queries, dim)).astype(np.float32)
    if form == "lognormal": items *= rng.lognormal(0, 0.5, size=(n, 1)).astype(np.float32)
    elif form == "one long": items[12345] *= 40
    elif form == "constant": items = np.sign(items) * np.float32(0.7)
    elif form == "infinite items": items[77, 5] = 1e6   # beyond the largest half
    elif form == "infinite query": q[7, 3] = 1e6
    elif form == "tied": items[:] = items[0]
    got = search_halves(pkg, dsx, items, q, k)
    if form == "infinite items":
        assert got is None   # searched as before
        return
    want = search_halves(pkg, dsx, items, q, k, 7)
    assert got[2] == (1 if form in ("infinite query", "tied") else 0)
    if got[2]:   # the same search
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        return
    # both within dim roundings of the exact sum (and the same bits: test_gpu_screen_bytes_halves.py)
    x, w = q.astype(np.float16).astype(np.float64), items.astype(np.float16).astype(np.float64)
    bound = dim * 2.0 ** -24 * np.sqrt((x ** 2).sum(axis=1))[:, None] * np.sqrt((w ** 2).sum(axis=1)).max()
    exact = np.einsum("qd,qkd->qk", x, w[got[1]])
    assert (np.abs(got[0] - exact) <= bound).all()
    assert (np.abs(got[0].astype(np.float64) - want[0]) <= 2 * bound).all()


def test_scratch_of_shorter_batches(pkg, dsx, rng):
    """What is reserved for batches that go in bytes holds shorter ones, which go in halves and need more."""
    batch, short, kdim, n, k = 4096, 1023, 768, 131072, 50
    print("[case] scratch of %d rows behind %d" % (short, batch), flush=True)
    dX, dW = dev(pkg, rng.integers(-3, 4, size=(short, kdim)).astype(np.float32)), dev(pkg, rng.integers(-3, 4, size=(kdim, n)).astype(np.float32))
    table = pkg.DeviceArray((dsx.dsx_screen_table_bytes(n, kdim),), np.uint8)
    keys, vals = pkg.DeviceArray((short, k), np.float32), pkg.DeviceArray((short, k), np.uint32)
    pkg.check(dsx.dsx_screen_table_build(dW.ptr, n, n, kdim, table.ptr))
    pkg.check(dsx.dsx_fc_topk_screened_reserve(0, batch, kdim, n, k))
    before, after = C.c_int(), C.c_int()
    pkg.check(dsx.dsx_get_memory_usage(C.byref(before), None))
    pkg.check(dsx.dsx_fc_topk_screened(dX.ptr, kdim, dW.ptr, table.ptr, None, short, kdim, n, LINEAR, None, k, keys.ptr, vals.ptr, 0, None, None, None, None))
    pkg.check(dsx.dsx_get_memory_usage(C.byref(after), None))
    assert after.value == before.value
    keys.numpy()
