"""Equal items and equal columns of a layer have equal scores, bit for bit, wherever they lie: results are ordered by score and then by
column, so that the lower of two equal ones always comes first.  The values are no integers: only sums in one order agree on them."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_kernels import dev
from test_gpu_screen import search

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def everything_screened(dsx):
    """Searches that are small for a test are screened too (by default only where that is expected to be faster)."""
    dsx.dsx_testing_set_screen(1)
    yield
    dsx.dsx_testing_set_screen(0)


def with_twins(rng, n, dim, front, back, pairs):
    """n normal rows, `pairs` of which are copied from the first `front` rows to somewhere behind row `back`, scaled so that many rows
    of the result hold them.  Returns the rows and twin[row] = the lower row of its pair (its own number: no pair)."""
    rows = rng.standard_normal((n, dim), dtype=np.float32) / np.float32(np.sqrt(dim))
    low = rng.choice(front, pairs, replace=False)
    high = back + rng.choice(n - back, pairs, replace=False)
    rows[low] *= np.float32(1.5)
    rows[high] = rows[low]
    twin = np.arange(n)
    twin[high] = low
    return rows, twin


def check_twins(scores, idx, twin):
    pairs = 0
    for r in range(len(idx)):
        at = {int(c): p for p, c in enumerate(idx[r])}
        for c, p in at.items():
            t = int(twin[c])
            if t == c:
                continue
            pairs += 1
            assert t in at, "row %d holds %d and not the equal %d before it" % (r, c, t)
            assert scores[r, at[t]] == scores[r, p] and at[t] < p, "row %d: %d and the equal %d" % (r, t, c)
    assert pairs > 0


# the first block of a screened search is 8,192 items; both sweeps (up to 256 components and more)
@pytest.mark.parametrize("n,queries,dim,k", [(70000, 512, 64, 50), (90003, 600, 300, 100), (66000, 520, 100, 200)])
def test_screened_search(pkg, dsx, rng, n, queries, dim, k):
    print("[case] equal items screened n=%d queries=%d dim=%d k=%d" % (n, queries, dim, k), flush=True)
    items, twin = with_twins(rng, n, dim, 8192, 8192, 3000)
    q = rng.standard_normal((queries, dim), dtype=np.float32)
    s, i = search(pkg, dsx, items, q, k)
    assert dsx.dsx_knn_last_search_path() == 1
    check_twins(s, i, twin)


# blocks of 1,024 items, the last one narrow (dim no multiple of 4: block by block); first block, then candidate ranges
@pytest.mark.parametrize("n,queries,dim,k,path", [(3 * 1024 + 100, 100, 130, 60, 0), (2 * 1024 + 40, 9, 70, 100, 0), (3 * 1024 + 8, 300, 258, 20, 0),
                                                  (20000, 70, 64, 100, 1), (9000, 100, 256, 50, 1)])
def test_search_in_blocks(pkg, dsx, rng, n, queries, dim, k, path):
    print("[case] equal items in blocks n=%d queries=%d dim=%d k=%d" % (n, queries, dim, k), flush=True)
    dsx.dsx_testing_set_knn_block_columns(1024)
    try:
        items, twin = with_twins(rng, n, dim, 1000, 1024 if path else n // 1024 * 1024, min(400, n % 1024 // 2) if path == 0 else 400)
        q = rng.standard_normal((queries, dim), dtype=np.float32)
        s, i = search(pkg, dsx, items, q, k)
        assert dsx.dsx_knn_last_search_path() == path
    finally:
        dsx.dsx_testing_set_knn_block_columns(0)
    check_twins(s, i, twin)


# screened with a bias; in fp32 ranges of the shapes whose first block other kernels would take
@pytest.mark.parametrize("batch,kdim,n,k,act,first,screened", [(2048, 64, 20000, 40, 3, 0, True), (640, 260, 30000, 100, 0, 0, True),
                                                               (100, 64, 6001, 40, 3, 256, False), (60, 128, 9000, 30, 1, 512, False)])
def test_layer(pkg, dsx, rng, batch, kdim, n, k, act, first, screened):
    print("[case] equal columns batch=%d kdim=%d n=%d k=%d act=%d" % (batch, kdim, n, k, act), flush=True)
    block = first or 2048
    W, twin = with_twins(rng, n, kdim, block, block, block // 3)
    W = np.ascontiguousarray(W.T)
    bias = None
    if screened:
        bias = (rng.standard_normal(n) * 0.1).astype(np.float32)
        bias = bias[twin]
    X = rng.standard_normal((batch, kdim), dtype=np.float32) * np.float32(0.5)
    dX, dW, db = dev(pkg, X), dev(pkg, W), dev(pkg, bias)
    keys, vals = pkg.DeviceArray((batch, k), np.float32), pkg.DeviceArray((batch, k), np.uint32)
    params = pkg.ActParams(0.01, 1.0, 1.0)
    dsx.dsx_testing_set_fc_topk_first_columns(first)
    dsx.dsx_fc_topk_flagged(1)
    try:
        pkg.check(dsx.dsx_fc_topk(dX.ptr, kdim, dW.ptr, pkg.ptr(db), batch, kdim, n, act, C.byref(params), k, keys.ptr, vals.ptr, 0, None, None,
                                  None, None))
        s, i = keys.numpy(), vals.numpy()
    finally:
        dsx.dsx_testing_set_fc_topk_first_columns(0)
    assert dsx.dsx_fc_topk_flagged(1) == 0
    check_twins(s, i, twin)
