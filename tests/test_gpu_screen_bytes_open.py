"""Searches in bytes that bytes cannot settle: tens of thousands of items whose scores lie closer together than the bytes' error, and not than that of
halves.  They are searched in halves then, as are those that follow, and not in fp32."""

import ctypes as C

import numpy as np
import pytest

from test_gpu_kernels import dev
from test_gpu_screen_bytes import LINEAR, default_switches, layer

pytestmark = pytest.mark.gpu

DIM = 128


def close_items(rng, n, queries, one_long):
    """30,000 items around one direction; their scores' deviation is 0.6 % of |x| |w|, a fifth of what bytes leave open, thrice what halves do."""
    base = rng.normal(size=DIM)
    base /= np.sqrt((base ** 2).sum())
    items = rng.normal(size=(n, DIM)) / np.sqrt(DIM)
    at = rng.permutation(n)[:30000]
    items[at] = base + items[at] * 0.068
    if one_long: items[np.setdiff1d(np.arange(n), at)[0]] *= -3
    return items.astype(np.float32), (base + rng.normal(size=(queries, DIM)) / np.sqrt(DIM) * 0.3).astype(np.float32)


@pytest.mark.parametrize("n,queries,k,one_long", [(70001, 300, 10, False), (70001, 300, 10, True), (300001, 70, 100, False), (32768, 600, 20, False)])
def test_search(pkg, dsx, rng, n, queries, k, one_long):
    print("[case] open search in bytes n=%d queries=%d k=%d one_long=%d" % (n, queries, k, one_long), flush=True)
    items, q = close_items(rng, n, queries, one_long)
    rows = (n + 7) // 8 * 8
    pkg.check(dsx.dsx_testing_set_screen_bytes(1))
    cm = np.full((DIM, rows), 1e30, dtype=np.float32)      # pad rows: never looked at
    cm[:, :n] = items.T
    dI, dQ = dev(pkg, cm), dev(pkg, q)
    room = pkg.DeviceArray((dsx.dsx_knn_workspace_bytes_prepared(rows, DIM, queries, k),), np.uint8)
    prepared = C.c_int(-1)
    pkg.check(dsx.dsx_knn_prepare(dI.ptr, rows, rows - n, DIM, queries, k, room.ptr, room.nbytes, C.byref(prepared)))
    assert prepared.value == (3 if one_long else 4)
    scores, idx = pkg.DeviceArray((queries, k), np.float32), pkg.DeviceArray((queries, k), np.uint32)

    def search(storage):
        pkg.check(dsx.dsx_knn_search_host(storage, dI.ptr, rows, rows - n, DIM, dQ.ptr, queries, k, scores.ptr, idx.ptr, None, None, room.ptr, room.nbytes, None))
        return scores.numpy(), idx.numpy(), dsx.dsx_knn_last_search_repeated(), dsx.dsx_knn_last_search_path()

    first, halves, fp32 = search(prepared.value), search(prepared.value + 5), search(5)
    assert first[2:] == (2, 1) and halves[2:] == (0, 1)
    assert np.array_equal(first[0], halves[0]) and np.array_equal(first[1], halves[1])
    # sums of 128 products, |q| |w| below 1.2 * 1.1, in two orders
    assert np.abs(first[0].astype(np.float64) - fp32[0]).max() <= 2 * DIM * 2.0 ** -24 * 1.32


def test_searches_that_follow(pkg, dsx, rng):
    """KnnExactGpu: one search in bytes for nothing, then ever more in halves."""
    from amazon_dsstne_amd import host_api
    lib = host_api.load_host_library()
    n, queries, k = 70001, 600, 10
    print("[case] searches behind an open one n=%d queries=%d k=%d" % (n, queries, k), flush=True)
    items, q = close_items(rng, n, queries, False)
    knn = lib.dsstne_knn_create(queries, k)
    try:
        assert lib.dsstne_knn_load(knn, items.ctypes.data, n, DIM, None) == 0
        scores, idx = np.empty((queries, k), np.float32), np.empty((queries, k), np.uint32)
        seen, results = [], []
        for _ in range(40):
            assert lib.dsstne_knn_search(knn, k, q.ctypes.data, queries, scores.ctypes.data, idx.ctypes.data) == 0
            seen.append(dsx.dsx_knn_last_search_repeated())
            results.append((scores.copy(), idx.copy()))
        assert set(seen) == {0, 2} and seen[0] == 2 and sum(s == 2 for s in seen) <= 6
        assert all(np.array_equal(results[0][0], s) and np.array_equal(results[0][1], i) for s, i in results)
    finally:
        lib.dsstne_knn_destroy(knn)


@pytest.mark.parametrize("n,batch,k", [(70001, 300, 10), (300001, 70, 100), (32768, 600, 20)])
def test_layer(pkg, dsx, rng, n, batch, k):
    """The rows of the first call are computed again; the second goes in halves, and neither tells its caller to store the layer."""
    print("[case] open layer in bytes n=%d batch=%d k=%d" % (n, batch, k), flush=True)
    items, X = close_items(rng, n, batch, False)
    W = np.ascontiguousarray(items.T)
    bias = np.zeros(n, np.float32)
    want = layer(pkg, dsx, X, W, bias, LINEAR, k, mode=2)
    assert want[2] == 0
    pkg.check(dsx.dsx_testing_set_screen_bytes(1))
    dX, dW, db = dev(pkg, X), dev(pkg, W), dev(pkg, bias)
    table = pkg.DeviceArray((dsx.dsx_screen_table_bytes(n, DIM),), np.uint8)
    keys, vals = pkg.DeviceArray((batch, k), np.float32), pkg.DeviceArray((batch, k), np.uint32)
    pkg.check(dsx.dsx_screen_table_build(dW.ptr, n, n, DIM, table.ptr))
    same = []
    for _ in range(12):
        pkg.check(dsx.dsx_fc_topk_screened(dX.ptr, DIM, dW.ptr, table.ptr, db.ptr, batch, DIM, n, LINEAR, None, k, keys.ptr, vals.ptr, 0, None, None, None, None))
        s, i = keys.numpy(), vals.numpy()
        # sums of 128 products, |x| |w| below 1.32, in two orders
        assert np.abs(s.astype(np.float64) - want[0]).max() <= 2 * DIM * 2.0 ** -24 * 1.32
        same.append(np.array_equal(s, want[0]) and np.array_equal(i, want[1]))
    # (fp32 sums have another order; 1, 4 and more calls in halves behind each in bytes)
    assert same == [False, True, False] + [True] * 4 + [False] + [True] * 4
    assert dsx.dsx_fc_topk_flagged_for(dW.ptr, 1) == 0
