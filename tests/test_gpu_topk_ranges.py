"""Top-K at the edges of its kernels: rows held in registers (topk_block_kernel), guided rows cut into parts, the merge of their lists,
and the nearest-neighbour search of few queries that uses them.  Everything but the last is compared bit for bit: a score matrix has one
right answer."""
import ctypes as C

import numpy as np
import pytest

from parity import assert_topk_exact
from test_gpu_kernels import dev, knn_case, run_filtered, run_guided, run_topk, segment_maxima
from test_oracle import random_csr

pytestmark = pytest.mark.gpu

# one row per workgroup: widths on both sides of 2, 8, 16 and 27 groups of 1,024 columns (a row may have six more than its groups),
# odd ones (rows at every alignment) and shorter than one group; k on both sides of 16 and at every list length; several workgroups per row
BLOCK = [(1030, 3, 3), (1025, 255, 16), (1024, 2041, 17), (1024, 2049, 64), (1024, 8185, 65), (1024, 8193, 128), (1024, 16377, 129),
         (1024, 16387, 10), (1024, 27637, 256), (1024, 27641, 100), (1024, 27648, 10), (1024, 27653, 200), (300, 27278, 128), (5, 100003, 256),
         (1, 8192, 256), (40, 16384, 1)]


@pytest.mark.parametrize("batch,width,k", BLOCK)
@pytest.mark.parametrize("filtered", [False, True])
def test_block_rows(pkg, dsx, orc, rng, batch, width, k, filtered):
    print("[case] block rows batch=%d width=%d k=%d filtered=%s" % (batch, width, k, filtered), flush=True)
    scores = rng.standard_normal((batch, width), dtype=np.float32)
    special = [np.float32(v) for v in (0.0, -0.0, np.finfo(np.float32).min, np.finfo(np.float32).max)]
    if not filtered:   # (times a listed column's zero an infinity is a NaN, which the oracle does not order)
        special += [np.float32(np.inf), np.float32(-np.inf)]
    rows = rng.integers(0, batch, 64)
    for n, r in enumerate(rows):
        scores[r, rng.integers(0, width)] = special[n % len(special)]
    for r, v in enumerate((1.0, -1.0, 0.0) if filtered else (1.0, -1.0, 0.0, -np.inf)):   # tied rows: nothing, or everything, reaches the bound
        if r < batch - 1:
            scores[batch - 1 - r] = v
    if filtered:
        start, end, fidx = random_csr(rng, batch, width, min(width, 300), empty_rows=(0,))
        keys, idx = run_filtered(pkg, dsx, scores, k, 0, None, start, end, fidx, None)
        rk, ri = orc.topk_filtered(scores, k, 0, None, start, end, fidx, None)
    else:
        keys, idx = run_topk(pkg, dsx, scores, k)
        rk, ri = orc.topk(scores, k)
    assert_topk_exact(keys, idx, rk, ri)


@pytest.mark.parametrize("width,k", [(2000, 10), (27278, 100), (9000, 200)])
def test_block_rows_with_nearly_everything_listed(pkg, dsx, orc, rng, width, k):
    """Fewer than k columns are left beside the listed ones, whose zeros then belong in the result."""
    batch = 1024
    print("[case] nearly everything listed width=%d k=%d" % (width, k), flush=True)
    scores = rng.random((batch, width), dtype=np.float32) + np.float32(0.01)
    start, end, cols = np.zeros(batch, np.uint64), np.zeros(batch, np.uint64), []
    for r in range(batch):
        listed = np.delete(np.arange(width, dtype=np.uint32), rng.integers(0, width, r % (2 * k))) if r % 64 == 1 else np.arange(r % 5, dtype=np.uint32)
        start[r] = end[r - 1] if r else 0
        cols.append(listed)
        end[r] = start[r] + len(listed)
    fidx = np.concatenate(cols)
    keys, idx = run_filtered(pkg, dsx, scores, k, 0, None, start, end, fidx, None)
    rk, ri = orc.topk_filtered(scores, k, 0, None, start, end, fidx, None)
    assert_topk_exact(keys, idx, rk, ri)


# guided rows cut into parts (few rows, wide ones), the smallest part, k <= 16 and above, and k in 65..128 where many rows make it pay
@pytest.mark.parametrize("batch,width,k", [(1, 32769, 10), (1, 1000003, 64), (2, 200001, 16), (4, 500000, 20), (64, 131073, 33), (40, 262145, 64),
                                           (260, 27278, 100), (300, 27279, 65), (230, 32768, 128)])
@pytest.mark.parametrize("form", ["random", "ties"])
@pytest.mark.parametrize("filtered", [False, True])
def test_guided_parts(pkg, dsx, orc, rng, batch, width, k, form, filtered):
    print("[case] guided parts batch=%d width=%d k=%d %s filtered=%s" % (batch, width, k, form, filtered), flush=True)
    scores = rng.standard_normal((batch, width), dtype=np.float32)
    if form == "ties":
        scores = np.minimum(scores, np.float32(1.0))                 # a sixth of every row ties at the top
        if not filtered:                                             # (run_filtered compares the matrix it sent with itself: no NaN)
            scores[0] = np.nan                                       # nothing to report
            if batch > 1:
                scores[-1] = -np.inf
    start = end = fidx = None
    if filtered:
        start, end, fidx = random_csr(rng, batch, width, 1500)
    keys, idx = run_guided(pkg, dsx, scores, k, segment_maxima(scores), 0, None, start, end, fidx, None)
    sk, si = run_filtered(pkg, dsx, scores, k, 0, None, start, end, fidx, None) if filtered else run_topk(pkg, dsx, scores, k)
    clean = slice(1, None) if form == "ties" and not filtered else slice(None)        # (the oracle orders no NaN)
    rk, ri = orc.topk_filtered(scores, k, 0, None, start, end, fidx, None) if filtered else orc.topk(scores, k)
    assert_topk_exact(keys[clean], idx[clean], rk[clean], ri[clean])
    assert_topk_exact(keys, idx, sk, si)


def test_guided_rows_under_capture(pkg, dsx, orc, rng):
    """Rows that would be cut into parts outside a capture: the graph uses no scratch of the library and gives the eager result on
    every replay, with new scores each time."""
    batch, width, k = 4, 100000, 10
    hip = C.CDLL("libamdhip64.so")
    dsx.dsx_stream.restype = C.c_void_p
    stream = C.c_void_p(dsx.dsx_stream())
    d, dm = pkg.DeviceArray((batch, width), np.float32), pkg.DeviceArray((batch, (width + 63) // 64), np.float32)
    keys, vals = pkg.DeviceArray((batch, k), np.float32), pkg.DeviceArray((batch, k), np.uint32)
    pkg.check(dsx.dsx_sync())
    graph, instance = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 2) == 0                 # relaxed
    rc = dsx.dsx_topk_guided(d.ptr, keys.ptr, vals.ptr, batch, width, k, dm.ptr, 64, 0, None, None, None, None, None)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    pkg.check(rc)
    nodes = C.c_size_t(0)
    assert hip.hipGraphGetNodes(graph, None, C.byref(nodes)) == 0 and nodes.value == 1
    assert hip.hipGraphInstantiate(C.byref(instance), graph, None, None, 0) == 0
    for _ in range(3):
        scores = rng.standard_normal((batch, width), dtype=np.float32)
        d.upload(scores)
        dm.upload(segment_maxima(scores))
        pkg.check(dsx.dsx_sync())
        assert hip.hipGraphLaunch(instance, stream) == 0
        pkg.check(dsx.dsx_sync())
        got = keys.numpy(), vals.numpy()
        rk, ri = orc.topk(scores, k)
        assert_topk_exact(got[0], got[1], rk, ri)
        ek, ei = run_guided(pkg, dsx, scores, k, segment_maxima(scores))
        assert_topk_exact(ek, ei, rk, ri)
    assert hip.hipGraphExecDestroy(instance) == 0 and hip.hipGraphDestroy(graph) == 0


def test_guided_rows_wider_than_one_part_under_capture(pkg, dsx, rng):
    """1,024 rows of more than 131,072 columns: one workgroup per row scans them, in a graph of one node without library scratch."""
    batch, width, k = 1024, 131137, 10
    hip = C.CDLL("libamdhip64.so")
    dsx.dsx_stream.restype = C.c_void_p
    stream = C.c_void_p(dsx.dsx_stream())
    scores = np.tile(rng.standard_normal((16, width), dtype=np.float32), (batch // 16, 1))
    scores[np.arange(batch), rng.integers(0, width, batch)] = np.float32(9.0)
    d, dm = dev(pkg, scores), dev(pkg, segment_maxima(scores))
    keys, vals = pkg.DeviceArray((batch, k), np.float32), pkg.DeviceArray((batch, k), np.uint32)
    pkg.check(dsx.dsx_sync())
    graph, instance = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 2) == 0                 # relaxed
    rc = dsx.dsx_topk_guided(d.ptr, keys.ptr, vals.ptr, batch, width, k, dm.ptr, 64, 0, None, None, None, None, None)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    pkg.check(rc)
    nodes = C.c_size_t(0)
    assert hip.hipGraphGetNodes(graph, None, C.byref(nodes)) == 0 and nodes.value == 1
    assert hip.hipGraphInstantiate(C.byref(instance), graph, None, None, 0) == 0
    want = run_topk(pkg, dsx, scores, k)
    for _ in range(2):
        keys.upload(np.zeros((batch, k), np.float32))
        pkg.check(dsx.dsx_sync())
        assert hip.hipGraphLaunch(instance, stream) == 0
        pkg.check(dsx.dsx_sync())
        assert_topk_exact(keys.numpy(), vals.numpy(), *want)
    assert hip.hipGraphExecDestroy(instance) == 0 and hip.hipGraphDestroy(graph) == 0


@pytest.mark.parametrize("items,queries,dim,k", [(200003, 1, 40, 20), (150001, 4, 128, 10), (70000, 64, 33, 64), (70000, 65, 33, 64),
                                                 (40000, 7, 16, 256), (500, 3, 16, 100)])
def test_knn_few_queries(pkg, dsx, orc, rng, items, queries, dim, k):
    """Small integer vectors: every score is exact whatever the order of the sum, so the result is the oracle's bit for bit,
    thousands of ties included."""
    print("[case] knn few queries items=%d queries=%d dim=%d k=%d" % (items, queries, dim, k), flush=True)
    it = rng.integers(-3, 4, size=(items, dim)).astype(np.float32)
    q = rng.integers(-3, 4, size=(queries, dim)).astype(np.float32)
    got_s, got_i, ref_s, ref_i, _ = knn_case(pkg, dsx, orc, it, q, k)
    assert np.array_equal(got_s, ref_s) and np.array_equal(got_i, ref_i)


def test_knn_search_returns_with_its_results(pkg, dsx, rng):
    """Block by block and without timers too: nothing is left on the stream when the call returns."""
    items, queries, dim, k = 1000000, 4, 64, 10
    hip = C.CDLL("libamdhip64.so")
    dsx.dsx_stream.restype = C.c_void_p
    stream = C.c_void_p(dsx.dsx_stream())
    table, q = pkg.DeviceArray((dim, items), np.float32), dev(pkg, rng.standard_normal((queries, dim), dtype=np.float32))
    scores, idx = pkg.DeviceArray((queries, k), np.float32), pkg.DeviceArray((queries, k), np.uint32)
    for _ in range(3):
        pkg.check(dsx.dsx_knn_search(table.ptr, items, 0, dim, q.ptr, queries, k, scores.ptr, idx.ptr, None, 0, None))
        assert dsx.dsx_knn_last_search_path() == 0 and hip.hipStreamQuery(stream) == 0


@pytest.mark.parametrize("items,queries,k", [(200000, 100, 200), (200000, 100, 129), (150001, 65, 100), (270011, 130, 256)])
def test_knn_segments_of_a_row_that_share_its_bound(pkg, dsx, orc, rng, items, queries, k):
    """Several workgroups per row raise one bound while their siblings read it, and thousands of items tie at every score: the order
    among them (lower item first) may not depend on who reads when."""
    print("[case] shared row bound items=%d queries=%d k=%d" % (items, queries, k), flush=True)
    dim = 8
    it = rng.integers(-1, 2, size=(items, dim)).astype(np.float32)
    q = rng.integers(-1, 2, size=(queries, dim)).astype(np.float32)
    got_s, got_i, ref_s, ref_i, _ = knn_case(pkg, dsx, orc, it, q, k)
    assert np.array_equal(got_s, ref_s) and np.array_equal(got_i, ref_i)


@pytest.mark.parametrize("items,most,fewer", [(500, 129, (128, 127, 64, 3)), (5000, 65, (64, 33, 1)), (20000, 43, (42, 7))])
@pytest.mark.parametrize("storage", ["fp32", "fp16", "split"])
def test_knn_workspace_of_a_batch_holds_smaller_ones(pkg, dsx, orc, rng, items, most, fewer, storage):
    """Fewer queries leave more lists each, which must not need more than a workspace sized for the whole batch."""
    dim, k = 24, 100
    rows = (items + 7) // 8 * 8
    suffix = "" if storage == "fp32" else "_f16" if storage == "fp16" else "_split"
    it = rng.integers(-3, 4, size=(items, dim)).astype(np.float32)
    cm = np.full((dim, rows), 50.0, dtype=np.float32)
    cm[:, :items] = it.T
    table = dev(pkg, cm)
    if storage == "fp16":
        made = pkg.DeviceArray((dsx.dsx_knn_f16_table_bytes(rows, dim),), np.uint8)
        pkg.check(dsx.dsx_knn_f16_convert_items(table.ptr, rows, rows - items, dim, made.ptr))
    elif storage == "split":
        made = pkg.DeviceArray((dsx.dsx_fc_split_bytes(rows, dim),), np.uint8)
        pkg.check(dsx.dsx_fc_split(table.ptr, rows, 1, rows, dim, made.ptr))
    else:
        made = table
    room = getattr(dsx, "dsx_knn_workspace_bytes" + suffix)(rows, dim, most, k)
    workspace = pkg.DeviceArray((room,), np.uint8)
    for queries in (most,) + fewer:
        print("[case] knn workspace items=%d most=%d queries=%d %s" % (items, most, queries, storage), flush=True)
        q = rng.integers(-3, 4, size=(queries, dim)).astype(np.float32)
        dq, scores, idx = dev(pkg, q), pkg.DeviceArray((queries, k), np.float32), pkg.DeviceArray((queries, k), np.uint32)
        pkg.check(getattr(dsx, "dsx_knn_search" + suffix)(made.ptr, rows, rows - items, dim, dq.ptr, queries, k, scores.ptr, idx.ptr,
                                                          workspace.ptr, room, None))
        rs, ri = orc.knn_search(cm, rows, rows - items, dim, q, k)
        assert np.array_equal(scores.numpy(), rs) and np.array_equal(idx.numpy(), ri)
