"""Searches and output layers screened by a table that the caller keeps: integer operands, whose scores are exact in fp32 and in f16 whatever
the order of the sums, so that the results are those of a full sort, ties by ascending column."""

import ctypes as C

import numpy as np
import pytest

from test_gpu_kernels import dev
from test_oracle import random_csr

pytestmark = pytest.mark.gpu


def best(full, k):
    """The k best of every row of whole numbers: score descending, then column ascending."""
    n = full.shape[1]
    key = full.astype(np.int64) * (1 << 32) + (n - 1 - np.arange(n, dtype=np.int64))
    part = np.argpartition(-key, k - 1, axis=1)[:, :k]
    part = np.take_along_axis(part, np.argsort(-np.take_along_axis(key, part, axis=1), axis=1), axis=1)
    return np.take_along_axis(full, part, axis=1), part.astype(np.uint32)


# every tile shape of the stored sums (up to 64, 128 and more rows; few and many tiles) and every form of the kernel that reads them, at the
# edges of its range; one case in ranges; filters that leave few blocks of 32 columns, or none, without a listed one
@pytest.mark.parametrize("batch,kdim,n,k,filtered", [(1, 32, 8192, 1, False), (48, 100, 27278, 20, True), (64, 128, 131072, 33, True),
                                                     (65, 64, 131073, 256, True), (128, 260, 8200, 32, True), (129, 512, 27278, 100, True),
                                                     (513, 96, 131073, 10, True), (300, 64, 140001, 50, True), (769, 32, 32769, 256, False),
                                                     (3, 36, 1048576, 40, True), (5, 32, 1048577, 7, True)])
def test_layer(pkg, dsx, rng, batch, kdim, n, k, filtered):
    print("[case] kept table layer batch=%d kdim=%d n=%d k=%d" % (batch, kdim, n, k), flush=True)
    X = rng.integers(-3, 4, size=(batch, kdim)).astype(np.float32)
    W = rng.integers(-3, 4, size=(kdim, n)).astype(np.float32)
    bias = rng.integers(-40, 41, size=n).astype(np.float32)
    start = end = fidx = None
    if filtered:
        start, end, fidx = random_csr(rng, batch, n, 300)
        all_but = np.delete(np.arange(n, dtype=np.uint32), np.arange(0, n, 23))   # of the last row: one column in 23 is left
        fidx = np.concatenate([fidx[:int(start[batch - 1])], all_but]).astype(fidx.dtype)
        end[batch - 1] = len(fidx)
    dX, dW, db, ds, de, dx = (dev(pkg, a) for a in (X, W, bias, start, end, fidx))
    table = pkg.DeviceArray((dsx.dsx_screen_table_bytes(n, kdim),), np.uint8)
    keys, vals = pkg.DeviceArray((batch, k), np.float32), pkg.DeviceArray((batch, k), np.uint32)
    pkg.check(dsx.dsx_screen_table_build(dW.ptr, n, n, kdim, table.ptr))
    pkg.check(dsx.dsx_fc_topk_screened(dX.ptr, kdim, dW.ptr, table.ptr, db.ptr, batch, kdim, n, 3, None, k, keys.ptr, vals.ptr, 0, None,
                                       pkg.ptr(ds), pkg.ptr(de), pkg.ptr(dx)))
    y = X @ W + bias
    if filtered:
        for b in range(batch):
            y[b, fidx[int(start[b]):int(end[b])]] = 0
    want_keys, want_vals = best(y, k)
    assert np.array_equal(keys.numpy(), want_keys)
    # (a zero of a listed column and one of another column tie; which of them is listed first is the path's own)
    differ = vals.numpy() != want_vals
    assert not differ[want_keys != 0].any()


@pytest.mark.parametrize("n,dim,most,k", [(65601, 768, 520, 100), (400003, 128, 4, 10), (270001, 187, 513, 33),
                                               (8192, 16, 70, 128), (8193, 19, 1, 1)])
def test_prepared_search(pkg, dsx, rng, n, dim, most, k):
    """Few queries, many, and the results in host memory."""
    print("[case] prepared search n=%d dim=%d queries=%d k=%d" % (n, dim, most, k), flush=True)
    items = rng.integers(-3, 4, size=(n, dim)).astype(np.float32)
    q = rng.integers(-3, 4, size=(most, dim)).astype(np.float32)
    rows = (n + 7) // 8 * 8
    cm = np.full((dim, rows), 1e30, dtype=np.float32)      # pad rows: never looked at
    cm[:, :n] = items.T
    dI, dQ = dev(pkg, cm), dev(pkg, q)
    room = pkg.DeviceArray((dsx.dsx_knn_workspace_bytes_prepared(rows, dim, most, k),), np.uint8)
    prepared = C.c_int(-1)
    pkg.check(dsx.dsx_knn_prepare(dI.ptr, rows, rows - n, dim, most, k, room.ptr, room.nbytes, C.byref(prepared)))
    assert prepared.value == 4
    rs, ri = best(q @ items.T, k)
    scores, idx = pkg.DeviceArray((most, k), np.float32), pkg.DeviceArray((most, k), np.uint32)
    host = C.c_void_p()
    pkg.check(dsx.dsx_malloc_host(C.byref(host), 8 * most * k))
    try:
        for queries in sorted({1, min(most, 64), most}):
            C.memset(host, 0, 8 * most * k)
            pkg.check(dsx.dsx_knn_search_host(prepared.value, dI.ptr, rows, rows - n, dim, dQ.ptr, queries, k, scores.ptr, idx.ptr, host.value,
                                              host.value + 4 * most * k, room.ptr, room.nbytes, None))
            words = np.ctypeslib.as_array(C.cast(host, C.POINTER(C.c_uint32)), (2, most * k)).copy()
            hs, hi = words[0].view(np.float32).reshape(most, k)[:queries], words[1].reshape(most, k)[:queries]
            assert np.array_equal(hs, rs[:queries]) and np.array_equal(hi, ri[:queries])
            assert np.array_equal(scores.numpy()[:queries], hs) and np.array_equal(idx.numpy()[:queries], hi)
    finally:
        dsx.dsx_free(host)


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("n,queries,k", [(5000, 3, 7), (20000, 700, 40), (150001, 520, 100)])
def test_results_in_host_memory(pkg, dsx, rng, storage, n, queries, k):
    """The last kernel of every other way of a search writes there too."""
    dim, rows = 64, (n + 7) // 8 * 8
    print("[case] host results storage=%d n=%d queries=%d k=%d" % (storage, n, queries, k), flush=True)
    items = rng.integers(-3, 4, size=(n, dim)).astype(np.float32)
    q = rng.integers(-3, 4, size=(queries, dim)).astype(np.float32)
    cm = np.zeros((dim, rows), dtype=np.float32)
    cm[:, :n] = items.T
    dI, dQ = dev(pkg, cm), dev(pkg, q)
    if storage == 1:
        table = pkg.DeviceArray((dsx.dsx_knn_f16_table_bytes(rows, dim),), np.uint8)
        pkg.check(dsx.dsx_knn_f16_convert_items(dI.ptr, rows, rows - n, dim, table.ptr))
    elif storage == 2:
        table = pkg.DeviceArray((dsx.dsx_fc_split_bytes(rows, dim),), np.uint8)
        pkg.check(dsx.dsx_fc_split(dI.ptr, rows, 1, rows, dim, table.ptr))
    else:
        table = dI
    scores, idx = pkg.DeviceArray((queries, k), np.float32), pkg.DeviceArray((queries, k), np.uint32)
    host = C.c_void_p()
    pkg.check(dsx.dsx_malloc_host(C.byref(host), 8 * queries * k))
    try:
        pkg.check(dsx.dsx_knn_search_host(storage, table.ptr, rows, rows - n, dim, dQ.ptr, queries, k, scores.ptr, idx.ptr, host.value,
                                          host.value + 4 * queries * k, None, 0, None))
        words = np.ctypeslib.as_array(C.cast(host, C.POINTER(C.c_uint32)), (2, queries, k)).copy()
        rs, ri = best(q @ items.T, k)
        assert np.array_equal(words[0].view(np.float32), rs) and np.array_equal(words[1], ri)
        assert np.array_equal(scores.numpy(), rs) and np.array_equal(idx.numpy(), ri)
    finally:
        dsx.dsx_free(host)


# tables whose pad rows lie across a width, or a product with the queries, at which whole rows stop being stored: laid out for the one side, searched
# on the other
@pytest.mark.parametrize("rows,padding,queries,k", [(131080, 8, 600, 10), (140000, 12000, 513, 33), (1048584, 16, 3, 20), (32400, 100, 8300, 10)])
def test_pad_rows_across_a_limit(pkg, dsx, rng, rows, padding, queries, k):
    print("[case] pad rows rows=%d padding=%d queries=%d k=%d" % (rows, padding, queries, k), flush=True)
    dim, n = 32, rows - padding
    items = rng.integers(-3, 4, size=(n, dim)).astype(np.float32)
    q = rng.integers(-3, 4, size=(queries, dim)).astype(np.float32)
    cm = np.full((dim, rows), 1e30, dtype=np.float32)
    cm[:, :n] = items.T
    dI, dQ = dev(pkg, cm), dev(pkg, q)
    room = pkg.DeviceArray((dsx.dsx_knn_workspace_bytes_prepared(rows, dim, queries, k),), np.uint8)
    prepared = C.c_int(-1)
    pkg.check(dsx.dsx_knn_prepare(dI.ptr, rows, padding, dim, queries, k, room.ptr, room.nbytes, C.byref(prepared)))
    assert prepared.value == 4
    scores, idx = pkg.DeviceArray((queries, k), np.float32), pkg.DeviceArray((queries, k), np.uint32)
    rows_looked_at = np.unique(np.concatenate([np.arange(min(queries, 40)), rng.integers(0, queries, 200), [queries - 1]]))
    rs, ri = best(q[rows_looked_at] @ items.T, k)
    # the kept table, a table made in the call, and the library's own workspace
    for storage, space in ((prepared.value, room), (0, room), (0, None)):
        scores.upload(np.zeros((queries, k), np.float32))
        pkg.check(dsx.dsx_knn_search_host(storage, dI.ptr, rows, padding, dim, dQ.ptr, queries, k, scores.ptr, idx.ptr, None, None,
                                          space.ptr if space else None, space.nbytes if space else 0, None))
        assert np.array_equal(scores.numpy()[rows_looked_at], rs) and np.array_equal(idx.numpy()[rows_looked_at], ri)
        if storage == prepared.value:   # (the other ways write over the table)
            assert dsx.dsx_knn_last_search_path() == 1


# more sums than are stored of whole tables, of a table no wider than a first block, which is all there is then
def test_large_batches_of_narrow_tables(pkg, dsx, rng):
    queries, n, dim, k = 66000, 16380, 16, 256
    print("[case] prepared search n=%d dim=%d queries=%d k=%d" % (n, dim, queries, k), flush=True)
    items = rng.integers(-3, 4, size=(n, dim)).astype(np.float32)
    q = rng.integers(-3, 4, size=(queries, dim)).astype(np.float32)
    rows, looked_at = n + 4, np.unique(np.concatenate([np.arange(20), rng.integers(0, queries, 200), np.arange(queries - 20, queries)]))
    cm = np.full((dim, rows), 1e30, dtype=np.float32)
    cm[:, :n] = items.T
    dI, dQ = dev(pkg, cm), dev(pkg, q)
    room = pkg.DeviceArray((dsx.dsx_knn_workspace_bytes_prepared(rows, dim, queries, k),), np.uint8)
    prepared = C.c_int(-1)
    pkg.check(dsx.dsx_knn_prepare(dI.ptr, rows, 4, dim, queries, k, room.ptr, room.nbytes, C.byref(prepared)))
    scores, idx = dev(pkg, np.zeros((queries, k), np.float32)), pkg.DeviceArray((queries, k), np.uint32)
    pkg.check(dsx.dsx_knn_search_host(prepared.value, dI.ptr, rows, 4, dim, dQ.ptr, queries, k, scores.ptr, idx.ptr, None, None, room.ptr, room.nbytes, None))
    rs, ri = best(q[looked_at] @ items.T, k)
    assert np.array_equal(scores.numpy()[looked_at], rs) and np.array_equal(idx.numpy()[looked_at], ri)

    print("[case] kept table layer batch=%d kdim=%d n=%d k=%d" % (queries, dim, n, k), flush=True)
    room.free()
    start, end, fidx = random_csr(rng, queries, n, 100)
    W, bias = np.ascontiguousarray(items.T), rng.integers(30, 41, size=n).astype(np.float32)
    dW, db, ds, de, dx = (dev(pkg, a) for a in (W, bias, start, end, fidx))
    table = pkg.DeviceArray((dsx.dsx_screen_table_bytes(n, dim),), np.uint8)
    pkg.check(dsx.dsx_screen_table_build(dW.ptr, n, n, dim, table.ptr))
    scores.upload(np.zeros((queries, k), np.float32))
    pkg.check(dsx.dsx_fc_topk_screened(dQ.ptr, dim, dW.ptr, table.ptr, db.ptr, queries, dim, n, 3, None, k, scores.ptr, idx.ptr, 0, None, ds.ptr,
                                       de.ptr, dx.ptr))
    y = q[looked_at] @ W + bias
    for at, b in enumerate(looked_at):
        y[at, fidx[int(start[b]):int(end[b])]] = 0
    rs, ri = best(y, k)
    assert np.array_equal(scores.numpy()[looked_at], rs)
    assert not (idx.numpy()[looked_at] != ri)[rs != 0].any()


def test_results_are_complete_without_events(pkg, dsx, rng):
    """The call returns with its results in host memory whether or not its stages can be timed."""
    n, dim, queries, k = 60000, 256, 2048, 100
    items = rng.integers(-3, 4, size=(n, dim)).astype(np.float32)
    q = rng.integers(-3, 4, size=(queries, dim)).astype(np.float32)
    dI, dQ = dev(pkg, np.ascontiguousarray(items.T)), dev(pkg, q)
    scores, idx = pkg.DeviceArray((queries, k), np.float32), pkg.DeviceArray((queries, k), np.uint32)
    host, elapsed = C.c_void_p(), (C.c_float * 2)()
    pkg.check(dsx.dsx_malloc_host(C.byref(host), 8 * queries * k))
    pkg.check(dsx.dsx_testing_set_screen(2))
    try:
        for none in (0, 1):
            pkg.check(dsx.dsx_testing_set_knn_no_events(none))
            C.memset(host, 0, 8 * queries * k)
            pkg.check(dsx.dsx_knn_search_host(0, dI.ptr, n, 0, dim, dQ.ptr, queries, k, scores.ptr, idx.ptr, host.value, host.value + 4 * queries * k, None,
                                              0, elapsed))
            words = np.ctypeslib.as_array(C.cast(host, C.POINTER(C.c_uint32)), (2, queries, k)).copy()
            assert dsx.dsx_knn_last_search_path() == 0
            assert np.array_equal(words[0].view(np.float32), scores.numpy()) and np.array_equal(words[1], idx.numpy()), "events: %d" % (1 - none)
        looked_at = rng.integers(0, queries, 50)
        rs, ri = best(q[looked_at] @ items.T, k)
        assert np.array_equal(words[0].view(np.float32)[looked_at], rs) and np.array_equal(words[1][looked_at], ri)
    finally:
        dsx.dsx_testing_reset()
        dsx.dsx_free(host)
