"""Searches in bytes of more rows than there is room for the words of: part after part, with the results of separate searches."""

import numpy as np
import pytest

from test_gpu_screen_bytes import LINEAR, default_switches, layer, search, search_halves
from test_oracle import random_csr

pytestmark = pytest.mark.gpu

# 36,900 bytes a row: 28,672 rows at once, so two parts, of 15,360 rows and of the others
N, DIM, ROWS = 32769, 16, 30001
CUTS = [0, 8000, 15360, 23001, ROWS]


def whole(rng, shape):
    return rng.integers(-3, 4, size=shape).astype(np.float32)


@pytest.mark.parametrize("halves", [False, True])
def test_search(pkg, dsx, rng, halves):
    print("[case] search in bytes, two parts, halves=%d" % halves, flush=True)
    items, q = whole(rng, (N, DIM)), whole(rng, (ROWS, DIM))
    find = search_halves if halves else search
    got = find(pkg, dsx, items, q, 3)
    for a, b in zip(CUTS, CUTS[1:]):
        want = find(pkg, dsx, items, np.ascontiguousarray(q[a:b]), 3)
        assert np.array_equal(got[0][a:b], want[0]) and np.array_equal(got[1][a:b], want[1])
        assert want[2] == 0
    assert got[2] == 0
    assert np.array_equal(got[0][::3001, 0], (q[::3001] @ items.T).max(axis=1))


def test_layer(pkg, dsx, rng):
    """Sums that start from biases, and a filter whose rows go by position."""
    print("[case] layer in bytes, two parts", flush=True)
    X, W, bias = whole(rng, (ROWS, DIM)), whole(rng, (DIM, N)), rng.integers(-40, 41, size=N).astype(np.float32)
    start, end, fidx = random_csr(rng, ROWS, N, 20)
    got = layer(pkg, dsx, X, W, bias, LINEAR, 3, (start, end, fidx))
    for a, b in zip(CUTS, CUTS[1:]):
        want = layer(pkg, dsx, np.ascontiguousarray(X[a:b]), W, bias, LINEAR, 3, (start[a:b], end[a:b], fidx))
        assert np.array_equal(got[0][a:b], want[0]) and np.array_equal(got[1][a:b], want[1])
