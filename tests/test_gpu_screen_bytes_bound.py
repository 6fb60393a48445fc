"""Searches in bytes: the bound by which words are left out holds where operands are nearly exact in bytes.  Operands whose scores are exact in fp32
whatever the order of the sums, against a full sort."""

import numpy as np
import pytest

from test_gpu_screen_bytes import LINEAR, default_switches, layer, search

pytestmark = pytest.mark.gpu

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
