"""fp16 storage: a query has the same results, bit for bit, in a search in bytes, in one that is not screened, and by itself."""

import numpy as np
import pytest

from test_gpu_screen_bytes import default_switches, search_halves

pytestmark = pytest.mark.gpu


# vectors of 1 to 65 pieces of 64 components, odd numbers of pieces among them; words looked through by either kernel; fewer and more candidates than the
# wavefronts of a row take at a time
@pytest.mark.parametrize("n,dim,queries,k", [(8192, 16, 70, 1), (32768, 64, 300, 128), (32769, 65, 600, 33), (70001, 130, 300, 50), (40000, 192, 513, 256), (131072, 300, 65, 10),
                                             (30001, 1000, 20, 100), (16384, 4096, 3, 100)])
def test_same_bits(pkg, dsx, rng, n, dim, queries, k):
    print("[case] halves in bytes, same bits n=%d dim=%d queries=%d k=%d" % (n, dim, queries, k), flush=True)
    items = rng.normal(size=(n, dim)).astype(np.float32)
    q = (rng.normal(size=(queries, dim)) * rng.lognormal(0, 1, size=(queries, 1))).astype(np.float32)
    got = search_halves(pkg, dsx, items, q, k)
    assert got[2] == 0
    for want in (search_halves(pkg, dsx, items, q, k, 7), search_halves(pkg, dsx, items, q[-1:], k, 7)):
        rows = len(want[0])
        assert np.array_equal(got[0][-rows:], want[0]) and np.array_equal(got[1][-rows:], want[1])
