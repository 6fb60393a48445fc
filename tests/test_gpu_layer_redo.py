"""Rows of a fused output layer that are computed again (layer_redo_kernel): tied scores by the thousand and listed columns' zeros, against
the two-call path bit for bit (every sum here is exact in any order)."""
import numpy as np
import pytest

from test_gpu_fctopk import ACT_LINEAR, ACT_RELU, ACT_SIGMOID, knobs, run_both  # noqa: F401
from test_oracle import random_csr

pytestmark = pytest.mark.gpu


# flagged rows: one, 31, 32, 33, all of them; widths on both sides of a span of 1,024 and a step of 128, several parts; sums no multiple
# of eight long; k at every list length
@pytest.mark.parametrize("batch,kdim,n,k,tied", [(70, 32, 9000, 50, 1), (70, 36, 6145, 64, 31), (100, 20, 6143, 65, 32), (100, 12, 8192, 128, 33),
                                                 (300, 8, 20001, 129, 290), (600, 4, 16511, 256, 600), (1100, 40, 7000, 1, 1100)])
@pytest.mark.parametrize("act", [ACT_RELU, ACT_LINEAR, ACT_SIGMOID])
@pytest.mark.parametrize("filtered", [False, True])
def test_tied_rows(pkg, dsx, orc, rng, knobs, batch, kdim, n, k, tied, act, filtered):  # noqa: F811
    print("[case] redo batch=%d kdim=%d n=%d k=%d tied=%d act=%d filtered=%s" % (batch, kdim, n, k, tied, act, filtered), flush=True)
    dsx.dsx_testing_set_fc_topk_first_columns(256)
    dsx.dsx_testing_set_fc_topk_candidate_capacity(2048)          # less than the widest range's ties, more than other rows need
    X = rng.integers(-2, 3, size=(batch, kdim)).astype(np.float32)
    W = rng.integers(-2, 3, size=(kdim, n)).astype(np.float32)
    X[rng.choice(batch, tied, replace=False)] = 0.0
    bias = np.where(rng.random(n) < 0.9, 40.0, -1.0).astype(np.float32)   # rows of zeros: nine tenths tie at the top (a sigmoid's 1)
    start = end = fidx = index = None
    if filtered:
        start, end, fidx = random_csr(rng, batch + 9, n + 20, 400, empty_rows=(3,))
        index = rng.permutation(batch + 9).astype(np.uint32)
    gk, gi, _, tk, ti = run_both(pkg, dsx, orc, X, W, bias, act, k, 4 if filtered else 0, index, start, end, fidx, "tied rows")
    assert np.array_equal(gi, ti) and np.array_equal(gk.view(np.uint32), tk.view(np.uint32))
    assert dsx.dsx_fc_topk_flagged(1) == 1


def test_saturated_layer_takes_milliseconds(pkg, dsx, rng):
    """Every row of a saturated layer flagged (the whole batch computed twice): a few times what the layer itself takes, where a
    wavefront per row took half a second."""
    import time
    batch, kdim, n, k = 4096, 1024, 27278, 10
    X = pkg.DeviceArray.from_numpy(np.abs(rng.standard_normal((batch, kdim), dtype=np.float32)))
    W = pkg.DeviceArray.from_numpy(np.abs(rng.standard_normal((kdim, n), dtype=np.float32)))
    keys, vals = pkg.DeviceArray((batch, k), np.float32), pkg.DeviceArray((batch, k), np.uint32)
    for rep in range(2):
        dsx.dsx_fc_topk_flagged(1)
        pkg.check(dsx.dsx_sync())
        t0 = time.perf_counter()
        pkg.check(dsx.dsx_fc_topk(X.ptr, kdim, W.ptr, None, batch, kdim, n, ACT_SIGMOID, None, k, keys.ptr, vals.ptr, 0, None, None, None, None))
        pkg.check(dsx.dsx_sync())
        ms = (time.perf_counter() - t0) * 1e3
    print("[time] saturated 4,096 x 1,024 x 27,278: %.2f ms" % ms, flush=True)
    assert dsx.dsx_fc_topk_flagged(1) == 1
    assert (keys.numpy() == 1.0).all() and np.array_equal(vals.numpy(), np.tile(np.arange(k, dtype=np.uint32), (batch, 1)))
    assert ms < 50.0                       # six times what it measures; 500 before
