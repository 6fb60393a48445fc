"""Searches in bytes: the bound by which words are left out holds where operands are nearly exact in bytes, where activations are flat, and where the
columns of the largest words have no score or a small one.  Operands whose scores are exact in fp32 whatever the order of the sums, against a full sort."""

import ctypes as C

import numpy as np
import pytest

from test_gpu_kept_tables import best
from test_gpu_kernels import dev
from test_gpu_screen_bytes import LINEAR, SIGMOID, default_switches, layer, search

pytestmark = pytest.mark.gpu

TANH, RELU = 1, 2

# words looked through by the kernel that scores, by one of their own, and by that with four times as many reads a lane
WIDTHS = [32768, 131072, 300001]


@pytest.mark.parametrize("n", WIDTHS)
@pytest.mark.parametrize("starts", [False, True])
def test_words_raised_by_their_places(pkg, dsx, n, starts):
    """A word may lie 46 units above its sum.  28 blocks of one-hot items score 0, in units of 1 / 127^2; six blocks in units eleven times as small score a
    little more, and hold all results."""
    dim, queries, k = 128, 300, 10
    print("[case] places in bytes n=%d starts=%d" % (n, starts), flush=True)
    small = np.float32(1 / np.sqrt(127.0))
    items = np.zeros((n, dim), dtype=np.float32)
    items[:, 0], items[:, 1] = -np.float32(0.707), np.float32(0.707)
    blocks = np.random.default_rng(5).permutation(n // 32)[:34]
    for b in blocks[:28]:
        items[b * 32:b * 32 + 32] = np.eye(dim, dtype=np.float32)[1 + np.arange(32)] * np.float32(1 + 7 / 1024)   # (sums that start from 0 have no bits there)
    for b in blocks[28:]:
        items[b * 32:b * 32 + 32] = small
        items[b * 32:b * 32 + 32, 0] = small / 127
    q = np.zeros((queries, dim), dtype=np.float32)
    q[:, 0] = 1
    if starts: scores, idx, told = layer(pkg, dsx, q, np.ascontiguousarray(items.T), np.zeros(n, np.float32), LINEAR, k)
    else: scores, idx, told = search(pkg, dsx, items, q, k)
    want = np.sort(np.concatenate([np.arange(b * 32, b * 32 + 32) for b in blocks[28:]]))[:k]
    assert (idx == want).all() and (scores == small / 127).all()
    assert told == 0


@pytest.mark.parametrize("n", WIDTHS)
@pytest.mark.parametrize("act", [SIGMOID, TANH, RELU])
def test_flat_activations(pkg, dsx, rng, n, act):
    """Some hundred columns a row of score 1, the sums of which lie far apart; and rows of fewer positive sums than results, the others all 0."""
    batch, kdim, k = 70, 64, 10
    print("[case] flat activation %d in bytes n=%d" % (act, n), flush=True)
    X = rng.permuted(np.tile(np.repeat([-2, 0, 2], [20, 24, 20]), (batch, 1)), axis=1).astype(np.float32)
    W = 2 * rng.integers(-1, 2, size=(kdim, n)).astype(np.float32)
    full = X @ W                                            # multiples of 4
    if act == RELU: level = np.sort(full, axis=1)[:, -6].max()
    else: level = np.sort(full, axis=1)[:, -200].max() - 18  # 200 columns of a row at 18 and more, none at 15 to 17 or 7 to 9 (where roundings decide)
    bias = np.full(n, -(level // 4 * 4 + 2), dtype=np.float32)
    z = full + bias[0]
    y = np.maximum(z, 0) if act == RELU else np.where(z >= (17 if act == SIGMOID else 9), np.float32(1), np.float32(0))
    if act != RELU: assert (y.sum(axis=1) >= k).all()
    keys, vals, _ = layer(pkg, dsx, X, W, bias, act, k)
    want_keys, want_vals = best(y, k)
    assert np.array_equal(vals, want_vals) and np.array_equal(keys, want_keys)


@pytest.mark.parametrize("n", WIDTHS)
@pytest.mark.parametrize("passing", [1, 25, 40])
def test_columns_that_always_pass(pkg, dsx, rng, n, passing):
    """Columns whose norms f16 does not hold, so that nothing is known of their scores, which are the lowest there are."""
    batch, kdim, k = 70, 64, 30
    print("[case] always passing columns in bytes n=%d passing=%d" % (n, passing), flush=True)
    X = rng.integers(0, 4, size=(batch, kdim)).astype(np.float32)
    X[:, 0] = 1
    W = rng.integers(-3, 4, size=(kdim, n)).astype(np.float32)
    bias = rng.integers(-40, 41, size=n).astype(np.float32)
    W[:, rng.permutation(n)[:passing]] = -10000.0
    keys, vals, told = layer(pkg, dsx, X, W, bias, LINEAR, k)
    want_keys, want_vals = best(X @ W + bias, k)
    assert np.array_equal(vals, want_vals) and np.array_equal(keys, want_keys)
    assert told == 0


@pytest.mark.parametrize("n", WIDTHS)
@pytest.mark.parametrize("missing,k", [(1, 1), (10, 10), (5, 10), (3000, 10)])
def test_items_that_are_no_numbers(pkg, dsx, rng, n, missing, k):
    """Items along one direction and queries against it: every score is far below 0, which is what the bytes of an item that is no number add up to."""
    dim, queries = 128, 300
    print("[case] NaN items in bytes n=%d missing=%d k=%d" % (n, missing, k), flush=True)
    items = (5 + rng.integers(-1, 2, size=(n, dim))).astype(np.float32)
    q = -rng.integers(1, 4, size=(queries, dim)).astype(np.float32)
    want_scores = q @ items.T
    gone = rng.permutation(n)[:missing]
    items[gone, rng.integers(0, dim, missing)] = np.nan
    want_scores[:, gone] = -100000.0
    scores, idx, repeated = search(pkg, dsx, items, q, k)
    want, at = best(want_scores, k)
    assert np.array_equal(idx, at) and np.array_equal(scores, want)
    assert repeated == 0


def test_words_of_columns_without_scores(pkg, dsx, rng):
    """The same items searched as if all of them were numbers: that what was listed is not enough shows in the scores, and the rows are given up."""
    n, dim, queries, k = 131072, 128, 300, 10
    print("[case] NaN items in bytes, taken for even", flush=True)
    items = (5 + rng.integers(-1, 2, size=(n, dim))).astype(np.float32)
    q = -rng.integers(1, 4, size=(queries, dim)).astype(np.float32)
    want_scores = q @ items.T
    gone = rng.permutation(n)[:k]
    items[gone, 3] = np.nan
    want_scores[:, gone] = -100000.0
    pkg.check(dsx.dsx_testing_set_screen_bytes(1))
    dI, dQ = dev(pkg, np.ascontiguousarray(items.T)), dev(pkg, q)
    room = pkg.DeviceArray((dsx.dsx_knn_workspace_bytes_prepared(n, dim, queries, k),), np.uint8)
    prepared = C.c_int(-1)
    pkg.check(dsx.dsx_knn_prepare(dI.ptr, n, 0, dim, queries, k, room.ptr, room.nbytes, C.byref(prepared)))
    assert prepared.value == 3
    scores, idx = pkg.DeviceArray((queries, k), np.float32), pkg.DeviceArray((queries, k), np.uint32)
    pkg.check(dsx.dsx_knn_search_host(4, dI.ptr, n, 0, dim, dQ.ptr, queries, k, scores.ptr, idx.ptr, None, None, room.ptr, room.nbytes, None))
    want, at = best(want_scores, k)
    assert np.array_equal(idx.numpy(), at) and np.array_equal(scores.numpy(), want)
    assert dsx.dsx_knn_last_search_repeated() != 0
