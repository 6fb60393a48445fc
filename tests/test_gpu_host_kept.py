"""Kept tables behind the C++ classes: what a program does between two searches or two top-Ks."""
import ctypes as C

import numpy as np
import pytest

from test_host_gpu import run_exe

pytestmark = pytest.mark.gpu


def test_knn_matrices_that_a_program_works_on_itself():
    rc, out = run_exe("test_knn_gpu")
    assert rc == 0 and "0 failed" in out, out[-3000:]


def network(synth, host_api, items, hidden, batch, batches=1, k=20):
    p = synth.autoencoder("kept-%d" % items, 5, items, [hidden], batch, k, batches=batches, zipf_s=1.0, nnz_mean=20, nnz_sigma=0.5, nnz_clip=(1, 200))
    return p, host_api.Network(p, max_k=k)


@pytest.mark.parametrize("items,hidden,batch", [(140000, 256, 8), (27278, 64, 300)])
def test_units_written_through_a_pointer_after_the_prediction(pkg, dsx, synth, items, hidden, batch):
    """A program that holds the hidden layer's buffer may write to it at any time after a prediction: the output layer is of the units that were
    there then."""
    from amazon_dsstne_amd import host_api
    p, net = network(synth, host_api, items, hidden, batch)
    try:
        net.bind_input()
        net.set_deferred_output(False)
        net.predict_batch(0)
        net.topk(p.k)
        want, _ = net.get_topk(p.batch)
        net.set_deferred_output(True)
        net.set_lanes(1)
        net.predict_batch(0)
        ptr = net.unit_buffer("Hidden1")
        net.predict_batch(0)
        ones = np.ones((p.batch, hidden), np.float32)
        pkg.check(dsx.dsx_memcpy_h2d(ptr, ones.ctypes.data, ones.nbytes))
        net.topk(p.k)
        got, _ = net.get_topk(p.batch)
        # sums of up to 256 products below 1 in another order: 1e-5 is far above their roundings
        assert np.abs(got - want).max() < 1e-5
    finally:
        net.close()


def test_vectors_without_components(pkg, dsx):
    """Loading takes what it took before there were kept tables."""
    from amazon_dsstne_amd import host_api
    lib = host_api.load_host_library()
    items = np.ones((9000, 32), np.float32)
    knn = lib.dsstne_knn_create(4, 5)
    try:
        assert lib.dsstne_knn_load(knn, items.ctypes.data, 9000, 0, None) == 0, lib.dsstne_last_error()
    finally:
        lib.dsstne_knn_destroy(knn)


@pytest.mark.parametrize("n,batch", [(20000, 32), (500000, 600)])
def test_tables_full_of_ties_stop_being_screened(pkg, dsx, rng, n, batch):
    """10,000 copies of one item: every search that wants it would be screened and done again.  Few are; other queries are screened as before."""
    from amazon_dsstne_amd import host_api
    lib = host_api.load_host_library()
    dim, k = 32, 10
    items = rng.integers(-3, 4, size=(n, dim)).astype(np.float32)
    items[5000:15000] = 3.0
    tied = np.ones((batch, dim), np.float32)
    apart = np.repeat(items[:1], batch, axis=0) * 2
    knn = lib.dsstne_knn_create(batch, k)
    try:
        assert lib.dsstne_knn_load(knn, items.ctypes.data, n, dim, None) == 0
        scores, idx = np.empty((batch, k), np.float32), np.empty((batch, k), np.uint32)
        best = {id(q): np.argsort(-(items @ q[0]), kind="stable")[:k] for q in (tied, apart)}

        def search(q):
            """Whether it was screened for nothing, and whether it was not screened at all."""
            assert lib.dsstne_knn_search(knn, k, q.ctypes.data, batch, scores.ctypes.data, idx.ctypes.data) == 0
            order = best[id(q)]
            assert np.array_equal(idx, np.repeat(order[None], batch, axis=0)) and np.array_equal(scores[0], items[order] @ q[0])
            return dsx.dsx_knn_last_search_repeated()

        assert search(apart) == 0
        assert sum(search(tied) for _ in range(200)) <= 9
        # one in a batch is enough
        assert sum(search(apart) for _ in range(70)) == 0
        mixed = apart.copy()
        mixed[batch - 1] = 1.0
        assert lib.dsstne_knn_search(knn, k, mixed.ctypes.data, batch, scores.ctypes.data, idx.ctypes.data) == 0
        assert dsx.dsx_knn_last_search_repeated() == 1 and np.array_equal(idx[batch - 1], best[id(tied)]) and np.array_equal(idx[0], best[id(apart)])
    finally:
        lib.dsstne_knn_destroy(knn)


def memory(dsx):
    gpu, cpu = C.c_int(), C.c_int()
    assert dsx.dsx_get_memory_usage(C.byref(gpu), C.byref(cpu)) == 0
    return gpu.value << 10


def test_the_first_top_k_makes_no_table(pkg, dsx, synth):
    """The weights' table is there once the input is bound, and not made in the middle of a request; nor is the scratch memory allocated there."""
    from amazon_dsstne_amd import host_api
    p, net = network(synth, host_api, 140000, 256, 8)
    try:
        net.bind_input()
        net.predict_batch(0)
        before = memory(dsx)
        net.topk(p.k)
        net.get_topk(p.batch)
        assert memory(dsx) - before < 100 << 20      # the table: 217 MB
        net.predict_batch(0)                         # (the other lane)
        net.topk(p.k)
        net.get_topk(p.batch)
        assert memory(dsx) == before
    finally:
        net.close()


@pytest.mark.parametrize("items,hidden,batch", [(140000, 256, 8), (27278, 128, 300)])
def test_weights_set_between_two_top_ks(pkg, dsx, synth, items, hidden, batch):
    """Every top-K is of the weights there are, whatever table is kept; and a table of new weights is made when they have stayed for a few of them,
    the top-Ks before being those of the stored layer, bit for bit."""
    from amazon_dsstne_amd import host_api
    p, net = network(synth, host_api, items, hidden, batch)
    stored = host_api.Network(p, max_k=p.k)
    rng = np.random.default_rng(8)

    def topk(n):
        n.predict_batch(0)
        n.topk(p.k)
        return n.get_topk(p.batch)[0]
    try:
        net.bind_input()
        stored.bind_input()
        stored.set_deferred_output(False)
        for change in range(4):
            if change:
                w = rng.permutation(p.weights[1])
                net.set_weights("Hidden1", "Output", weights=w)
                stored.set_weights("Hidden1", "Output", weights=w)
            want = topk(stored)
            got = [topk(net) for _ in range(12 if change < 3 else 2)]
            # sums of up to 256 products below 1 in another order: 1e-5 is far above their roundings
            assert max(np.abs(g - want).max() for g in got) < 1e-5
            assert np.array_equal(got[0], want) == (change > 0)
            assert not (change < 3 and np.array_equal(got[-1], want))
    finally:
        stored.close()
        net.close()


@pytest.mark.parametrize("change", ["split products", "stored output"])
def test_a_table_that_is_not_used_is_given_back(pkg, dsx, synth, change):
    from amazon_dsstne_amd import host_api
    p, net = network(synth, host_api, 140000, 256, 8)
    try:
        net.bind_input()
        net.predict_batch(0)
        net.topk(p.k)
        net.get_topk(p.batch)
        before = memory(dsx)
        want = net.get_topk(p.batch)
        if change == "split products":
            net.set_split_products(True)             # (the weights' planes, 215 MB, come in its place)
            net.predict_batch(0)
            net.topk(p.k)
            assert memory(dsx) - before < 10 << 20
        else:
            net.set_deferred_output(False)
            assert before - memory(dsx) > 200 << 20
        net.set_split_products(False)
        net.set_deferred_output(True)
        assert before - memory(dsx) < 10 << 20       # (it is used again)
        net.predict_batch(0)
        net.topk(p.k)
        assert all(np.array_equal(a, b) for a, b in zip(want, net.get_topk(p.batch)))
    finally:
        net.close()
