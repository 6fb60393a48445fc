"""Kept tables with operands that f16 rounds: what is screened out must be what cannot be a result, at the edges of what the error allows, for
norms that lie decades apart, in every form of the search (few rows and many, sums stored and in ranges)."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_kernels import dev
from test_gpu_screen import check_against_float64
from test_oracle import random_csr

pytestmark = pytest.mark.gpu


def some(rng, rows, most=40):
    """Rows that the results are looked at of: the first, the last and others."""
    return np.unique(np.concatenate([[0, rows - 1], rng.integers(0, rows, most)]))


def layer(pkg, dsx, X, W, bias, k, act, csr=(None, None, None)):
    batch, kdim, n = len(X), W.shape[0], W.shape[1]
    dX, dW, db, ds, de, dx = (dev(pkg, a) for a in (X, W, bias) + tuple(csr))
    table = pkg.DeviceArray((dsx.dsx_screen_table_bytes(n, kdim),), np.uint8)
    keys, vals = pkg.DeviceArray((batch, k), np.float32), pkg.DeviceArray((batch, k), np.uint32)
    pkg.check(dsx.dsx_screen_table_build(dW.ptr, n, n, kdim, table.ptr))
    pkg.check(dsx.dsx_fc_topk_screened(dX.ptr, X.shape[1], dW.ptr, table.ptr, pkg.ptr(db), batch, kdim, n, act, None, k, keys.ptr, vals.ptr, 0, None,
                                       pkg.ptr(ds), pkg.ptr(de), pkg.ptr(dx)))
    return keys.numpy(), vals.numpy()


# few rows, up to 128, more, a table wider than 131,072 columns for few rows and for many (in ranges)
@pytest.mark.parametrize("batch,n", [(1, 131073), (48, 30000), (65, 131072), (129, 27278), (300, 140000), (600, 140000)])
@pytest.mark.parametrize("form", ["results round down", "others round up"])
def test_errors_as_large_as_they_get(pkg, dsx, rng, batch, n, form):
    """All components lie next to the middle between two halves.  'results round down': three long columns whose products cancel, every one of which
    rounds the wrong way: in f16 they lie 3 % below columns that they are above, and with half of their error added to their sums they would be lost.  'others
    round up': it is the others that are long, and with two thirds of what is taken off their sums the bound would lie above the results."""
    print("[case] kept table %s batch=%d n=%d" % (form, batch, n), flush=True)
    kdim, k, tiny = 128, 20, 2.0 ** -20
    up, down = 1 + 2.0 ** -11 + tiny, 1 + 2.0 ** -11 - tiny      # rounded to halves 1 + 2^-10 and 1
    scale = 2.0 ** rng.integers(-3, 4, batch)
    a, b = np.arange(kdim) % 2 == 0, np.arange(kdim) % 2 == 1    # 64 components each
    few = np.flatnonzero(a)[:60]
    W = (rng.standard_normal((kdim, n)) * 0.2).astype(np.float32)
    short, long = np.zeros(kdim), np.zeros(kdim)
    if form == "results round down":
        x = np.where(a, up, down)
        short[a] = up                                            # 64.1 in f16, 64.06
        long[b], long[few] = 16 * down, -16 * up                 # 62.1 in f16, 64.06
        best, other = long, short
    else:
        x = np.where(a, down, up)
        short[a] = down                                          # 64.0 in f16, 64.06
        long[b], long[few] = 16 * up, -16 * down                 # 66.1 in f16, 64.06
        best, other = short, long
    at = rng.permutation(n // 128)[:3 + 6 * k] * 128              # 64 columns and a block of 32 of their own
    lift = (best @ x - other @ x) - 0.03                          # the others end up 0.03 below the results, each by a little more than the one before
    W[:, at[:3]] = best[:, None]
    W[:, at[3:]] = other[:, None]
    W[0 if form == "results round down" else 1, at[3:]] += ((lift - np.arange(6 * k) * 2e-3) / x[0 if form == "results round down" else 1]).astype(np.float32)
    X = (x * scale[:, None]).astype(np.float32)
    s, i = layer(pkg, dsx, X, W, None, k, 3)
    at_rows = some(rng, batch)
    X, s, i, scale = X[at_rows], s[at_rows], i[at_rows], scale[at_rows]
    full = (X.astype(np.float64) @ W.astype(np.float64)) / scale[:, None]
    # 128 roundings of the sums of products at most, of 2^-24 of the 1,984 that the long columns' products add up to: half of what the results are ahead
    check_against_float64(s / scale[:, None], i, full, k, 128 * 1984 * 2.0 ** -24)
    assert all(set(at[:3].tolist()) <= set(r) for r in i.tolist())


@pytest.mark.parametrize("batch,n,kdim,k,act", [(1, 100003, 128, 50, 0), (48, 140001, 100, 20, 0), (65, 131073, 260, 10, 3), (129, 27278, 512, 100, 0),
                                                (300, 131072, 64, 40, 1), (600, 140000, 96, 100, 0)])
def test_norms_decades_apart(pkg, dsx, rng, batch, n, kdim, k, act):
    print("[case] kept table, norms apart batch=%d kdim=%d n=%d k=%d act=%d" % (batch, kdim, n, k, act), flush=True)
    X = np.maximum(rng.standard_normal((batch, kdim), dtype=np.float32), 0)
    W = rng.standard_normal((kdim, n), dtype=np.float32) * np.float32(1 / np.sqrt(kdim))
    W *= (10.0 ** rng.uniform(-4, 0, n)).astype(np.float32)
    bias = (rng.standard_normal(n) - 3).astype(np.float32)
    start, end, fidx = random_csr(rng, batch, n, 300)
    s, i = layer(pkg, dsx, X, W, bias, k, act, (start, end, fidx))
    at_rows = some(rng, batch)
    s, i = s[at_rows], i[at_rows]
    z = X[at_rows].astype(np.float64) @ W.astype(np.float64) + bias
    y = {0: lambda v: 1 / (1 + np.exp(-v)), 1: np.tanh, 3: lambda v: v}[act](z)
    for r, b in enumerate(at_rows):
        y[r, fidx[int(start[b]):int(end[b])]] *= 0.0
    # sums of kdim products and the bias, |x| |w| + |b| below 40 here: kdim roundings of 2^-24 of that at the very most, 1e-6 for the activations' own
    # error; slopes are at most 1
    check_against_float64(s, i, y, k, (kdim + 8) * 40 * 2.0 ** -24 / 8 + 1e-6)


@pytest.mark.parametrize("batch,n", [(3, 30000), (100, 140000), (600, 140000)])
def test_weights_that_are_no_numbers(pkg, dsx, rng, batch, n):
    """NaN, infinite and very large weights in a kept table."""
    print("[case] kept table, NaN and infinities batch=%d n=%d" % (batch, n), flush=True)
    kdim, k = 64, 30
    X = np.abs(rng.standard_normal((batch, kdim), dtype=np.float32)) + np.float32(0.01)
    W = rng.standard_normal((kdim, n), dtype=np.float32)
    W[5, 7::13] = np.nan
    W[9, [1000, 20001, n - 1]] = np.inf
    W[9, [1001, 20002]] = -np.inf
    W[:, [3, n // 2]] *= np.float32(1e6)
    W[:, 12000] = np.float32(6e4)      # (components that f16 holds, a norm that it does not)
    s, i = layer(pkg, dsx, X, W, None, k, 3)
    at_rows = some(rng, batch)
    X, s, i = X[at_rows], s[at_rows], i[at_rows]
    # (infinite scores as a number above all others, and below)
    full = np.nan_to_num(X.astype(np.float64) @ W.astype(np.float64), nan=-1e30, posinf=1e12, neginf=-1e12)
    large = np.take_along_axis(np.abs(full), i.astype(np.int64), axis=1) > 1e4
    assert (i[:, :2] != i[:, 1:3]).all() and all({1000, 20001, n - 1} - set(range(7, n, 13)) <= set(r) for r in i.tolist())
    at = np.take_along_axis(full, i.astype(np.int64), axis=1)
    got = np.nan_to_num(s.astype(np.float64), posinf=1e12)
    norm = np.linalg.norm(X.astype(np.float64), axis=1)[:, None]
    # large scores in units of themselves (their products are of one sign or the column's norm is what 64 of them come to), the others as elsewhere
    assert np.abs(got - at)[large].max() <= 1e-4 * np.abs(at[large]).max()
    assert np.abs((got - at) / norm)[~large].max() <= kdim * 2.0 ** -24 * 12
    want = np.sort(full, axis=1)[:, ::-1][:, :k]
    small = want < 1e4
    assert np.abs(((np.sort(at, axis=1)[:, ::-1] - want) / norm)[small]).max() <= kdim * 2.0 ** -24 * 12
    assert (want[~small] == np.sort(at, axis=1)[:, ::-1][~small]).all()


# norms apart and close together; sums stored; in ranges, with queries in registers and in LDS
@pytest.mark.parametrize("n,dim,queries,k,storage", [(70001, 96, 40, 30, 3), (140001, 100, 600, 50, 3), (140001, 300, 600, 20, 3), (70001, 96, 40, 30, 4),
                                                     (140001, 100, 600, 50, 4), (140001, 300, 600, 20, 4), (300007, 64, 1030, 10, 4)])
def test_prepared_searches(pkg, dsx, rng, n, dim, queries, k, storage):
    print("[case] prepared search n=%d dim=%d queries=%d k=%d storage=%d" % (n, dim, queries, k, storage), flush=True)
    items = rng.standard_normal((n, dim), dtype=np.float32)
    items /= np.linalg.norm(items, axis=1, keepdims=True)
    if storage == 3:
        items *= (10.0 ** rng.uniform(-1.2, 0, n)).astype(np.float32)[:, None]
    q = rng.standard_normal((queries, dim), dtype=np.float32) * (10.0 ** rng.uniform(-2, 2, queries)).astype(np.float32)[:, None]
    rows = (n + 7) // 8 * 8
    cm = np.full((dim, rows), 1e30, dtype=np.float32)      # pad rows: never looked at
    cm[:, :n] = items.T
    dI, dQ = dev(pkg, cm), dev(pkg, q)
    room = pkg.DeviceArray((dsx.dsx_knn_workspace_bytes_prepared(rows, dim, queries, k),), np.uint8)
    prepared = C.c_int(-1)
    pkg.check(dsx.dsx_knn_prepare(dI.ptr, rows, rows - n, dim, queries, k, room.ptr, room.nbytes, C.byref(prepared)))
    assert prepared.value == storage
    scores, idx = pkg.DeviceArray((queries, k), np.float32), pkg.DeviceArray((queries, k), np.uint32)
    pkg.check(dsx.dsx_knn_search_host(storage, dI.ptr, rows, rows - n, dim, dQ.ptr, queries, k, scores.ptr, idx.ptr, None, None, room.ptr, room.nbytes, None))
    assert dsx.dsx_knn_last_search_path() == 1 and dsx.dsx_knn_last_search_repeated() == 0
    at_rows = some(rng, queries)
    q, s, i = q[at_rows], scores.numpy()[at_rows], idx.numpy()[at_rows]
    full = q.astype(np.float64) @ items.astype(np.float64).T
    scale = np.linalg.norm(q.astype(np.float64), axis=1)[:, None]
    # dim products, each rounding at most 2^-24 of |q| |w|, |w| at most 1
    check_against_float64(s / scale, i, full / scale, k, dim * 2.0 ** -24)


def test_a_first_block_whose_best_columns_are_listed(pkg, dsx, rng):
    """Every row's filter lists the 144 best of the first 8,192 columns: the bound that is left lets one column in fifty of the next range pass, which is
    within what the lists hold."""
    batch, n, kdim, k = 600, 600000, 32, 10
    print("[case] kept table, listed first block batch=%d kdim=%d n=%d k=%d" % (batch, kdim, n, k), flush=True)
    X = np.maximum(rng.standard_normal((batch, kdim), dtype=np.float32), 0)
    W = rng.standard_normal((kdim, n), dtype=np.float32) * np.float32(1 / np.sqrt(kdim))
    bias = (rng.standard_normal(n) * 0.5 - 4).astype(np.float32)
    own = np.sort(np.argpartition(-(X @ W[:, :8192] + bias[:8192]), 144, axis=1)[:, :144], axis=1).astype(np.uint32)
    start = np.arange(batch, dtype=np.uint64) * 144
    dsx.dsx_fc_topk_flagged(1)
    s, i = layer(pkg, dsx, X, W, bias, k, 0, (start, start + 144, own.reshape(-1)))
    assert dsx.dsx_fc_topk_flagged(0) == 0
    at_rows = some(rng, batch, 20)
    y = 1 / (1 + np.exp(-(X[at_rows].astype(np.float64) @ W.astype(np.float64) + bias)))
    for r, b in enumerate(at_rows):
        y[r, own[b]] = 0
    # sums of kdim products and the bias, |x| |w| + |b| below 40: as above; the slope is a quarter at most
    check_against_float64(s[at_rows], i[at_rows], y, k, (kdim + 8) * 40 * 2.0 ** -24 / 8 + 1e-6)
