"""What the framework's performance is measured on: the work a user has it do, from one request to full batches.

Four kinds of work, each through the public entry points:

  serve   one request at a time: the rows arrive as host arrays (NNDataSet::LoadSparseData), one PredictBatch, one top-K, the
          results read back — what a service around the reference's JNI `predict` does;
  sweep   recommendations for a whole resident data set, batch after batch, the results of a batch collected while the next one
          runs — what the `predict` tool does; the last batch is usually a short one;
  knn     exact nearest neighbours of a batch of query vectors among the loaded items (KnnExactGpu::search), host arrays in and out;
  rank    the k best entries of every row of a score matrix that is already on the device (kCalculateTopK and its filtered and
          key/value forms), for programs that produce their scores themselves.

Weights are scaled as a trained network's are (unit-sized activations, output biases that follow the items' popularity, so that
most scores are small and few tie); items follow a Zipf law, so that popular ones are shared by many rows.
"""
import importlib
import importlib.util
import math
import os
import sys

import numpy as np
import torch


def package():
    """The package directory has a hyphen in its name and is loaded by path from the working folder."""
    name = "amazon_dsstne_amd"
    if name not in sys.modules:
        folder = os.path.join(os.getcwd(), "amazon-dsstne_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(folder, "__init__.py"), submodule_search_locations=[folder])
        sys.modules[name] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[name])
        importlib.import_module(name + ".host_api")
    return sys.modules[name]


ACTIVATIONS = {"sigmoid": 0, "tanh": 1, "relu": 2, "linear": 3, "softmax": 7}
VALUES = {"boolean": None, "float": np.float32, "double": np.float64, "uchar": np.uint8, "int": np.int32}


def network_case(name, kind, items, hidden, depth, batch, rows, k, nnz, zipf=1.0, act="relu", out="sigmoid", values="boolean",
                 weighted=False, indexed=False, filtered=True, split=False):
    c = dict(kind=kind, items=items, hidden=hidden, depth=depth, batch=batch, rows=rows, k=k, nnz=nnz, zipf=zipf, act=act, out=out,
             values=values, weighted=weighted, indexed=indexed, filtered=filtered, split=split)
    return dict(c, name=name) if name else c


def knn_case(name, items, dim, queries, k, storage):
    c = dict(kind="knn", items=items, dim=dim, queries=queries, k=k, storage=storage)
    return dict(c, name=name) if name else c


def rank_case(name, batch, width, k, form):
    c = dict(kind="rank", batch=batch, width=width, k=k, form=form)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a small shop's autoencoder, 32 visitors per request: launches and latency
        network_case("serve_tiny", "serve", 1024, 64, 1, 32, 32, 10, 16, zipf=0.0),
        # one visitor of a 27,278-item catalogue (the headline network): latency of every stage for a single row
        network_case("serve_one_row", "serve", 27278, 128, 3, 1, 1, 10, 144),
        # a request of 64 users to a softmax recommender over ratings with per-user weights
        network_case("serve_softmax_ratings", "serve", 27278, 512, 2, 64, 64, 20, 100, act="tanh", out="softmax", values="float", weighted=True),
        # a few visitors of a large catalogue: the output layer's weights have to be read for 8 rows
        network_case("serve_large_catalogue", "serve", 500000, 256, 1, 8, 8, 50, 50, zipf=1.1),
        # recommendations for everybody, headline network: batches of 1,024, the last one short
        network_case("sweep_catalogue", "sweep", 27278, 128, 3, 1024, 7900, 10, 144),
        # the reference's benchmark network (three hidden layers of 1,024, sigmoid), batches of 256, the predict tool's 100 results
        network_case("sweep_benchmark_net", "sweep", 27278, 1024, 3, 256, 1000, 100, 144, act="sigmoid"),
        # ratings of shuffled users (indexed data set), batches of 4,096 through two hidden layers of 1,024
        network_case("sweep_analog_indexed", "sweep", 27278, 1024, 2, 4096, 6000, 10, 144, values="float", indexed=True),
        # a million items, 512 hidden units, 4,096 users: the largest layer one device is asked for
        network_case("sweep_million_items", "sweep", 1000000, 512, 1, 4096, 4096, 100, 50, zipf=1.1),
        # nearest neighbours of a large batch of queries, and the same with halves as storage
        knn_case("knn_batch", 1000000, 128, 4096, 100, "fp32"),
        knn_case("knn_batch_fp16", 1000000, 128, 4096, 100, "fp16"),
        # an online lookup: a handful of queries, the table is read once for all of them
        knn_case("knn_lookup", 1000000, 128, 4, 20, "fp32"),
        # scores of one's own over the catalogue, the 128 best per row without the items the row already has
        rank_case("rank_scores", 1024, 27278, 128, "filtered"),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _hidden(rng, hi):
    h = _log(rng, 32, max(33, hi))
    return h if rng.random() < 0.25 else max(32, h // 32 * 32)   # layer widths are mostly round numbers


def draw(rng):
    kind = rng.choice(("serve", "serve", "sweep", "sweep", "knn", "rank"))
    if kind == "knn":
        dim, queries = _log(rng, 16, 256), _log(rng, 1, 4096)
        return knn_case(None, _log(rng, 20000, 1000000), dim, queries, _log(rng, 1, 128), rng.choice(("fp32", "fp32", "fp16", "fp32-split")))
    if kind == "rank":
        width = _log(rng, 1000, 200000)
        return rank_case(None, _log(rng, 1, min(2048, 60000000 // width)), width, _log(rng, 1, 256),
                         rng.choice(("plain", "filtered", "filtered", "kv")))
    if kind == "serve":
        items, batch = _log(rng, 1000, 500000), _log(rng, 1, 256)
        rows, depth, values, indexed = batch, rng.randint(1, 3), rng.choice(("boolean", "boolean", "float", "uchar")), False
    else:
        items, batch = _log(rng, 2000, 60000), _log(rng, 128, 4096)
        rows, depth = batch * rng.randint(1, 4) - rng.randint(0, batch // 2), rng.randint(1, 3)
        values, indexed = rng.choice(("boolean", "boolean", "float", "double", "int")), rng.random() < 0.3
    out = "softmax" if rng.random() < 0.15 else "sigmoid"
    return network_case(None, kind, items, _hidden(rng, min(1024, 130000000 // items)), depth, batch, rows, _log(rng, 1, 128),
                        _log(rng, 8, max(9, min(200, items // 40))), zipf=rng.choice((0.8, 1.0, 1.1)), act=rng.choice(("relu", "relu", "sigmoid", "tanh")),
                        out=out, values=values, weighted=rng.random() < 0.2, indexed=indexed, filtered=rng.random() < 0.8,
                        split=kind == "sweep" and rng.random() < 0.2)


# ------------------------------------------------------------------------------------------------------------------- inputs

def item_law(items, zipf):
    """Probability of every item: Zipf over its rank."""
    p = 1.0 / np.arange(1, items + 1, dtype=np.float64) ** zipf
    return p / p.sum()


def sparse_rows(rng, rows, items, nnz, p):
    """CSR rows of distinct ascending columns: lognormal numbers of items (sigma 1), drawn by popularity; repeated draws of an
    item within a row count once."""
    counts = np.clip(np.rint(rng.lognormal(math.log(nnz) - 0.5, 1.0, rows)), 1, min(2000, items // 8)).astype(np.int64)
    cdf = np.cumsum(p)
    drawn = np.minimum(np.searchsorted(cdf, rng.random(int(counts.sum())) * cdf[-1]), items - 1)
    shuffled = np.random.default_rng(items).permutation(items)[drawn]
    cells = torch.from_numpy(np.repeat(np.arange(rows, dtype=np.int64), counts) * items + shuffled).cuda().unique().cpu().numpy()
    end = np.searchsorted(cells, (np.arange(rows, dtype=np.int64) + 1) * items).astype(np.uint64)
    start = np.concatenate([np.zeros(1, np.uint64), end[:-1]])
    return start, end, (cells % items).astype(np.uint32)


class Problem:
    """A chain network and its sparse input, in the form the Python binding takes."""

    def __init__(self, case, seed):
        pkg = package()
        rng = np.random.default_rng(seed)
        gen = torch.Generator(device="cuda").manual_seed(seed)
        items, rows = case["items"], case["rows"]
        self.name = "%s-%d" % (case["kind"], items)
        self.batch, self.k = case["batch"], case["k"]
        self.widths = [items] + [case["hidden"]] * case["depth"] + [items]
        self.acts = [ACTIVATIONS[case["act"]]] * case["depth"] + [ACTIVATIONS[case["out"]]]
        p = item_law(items, case["zipf"])
        self.weights, self.biases = [], []
        for i in range(len(self.widths) - 1):
            last = i == len(self.widths) - 2
            # a unit's input is a sum over the row's items in the first layer, over all units of the layer before in the others
            fan_in = case["nnz"] if i == 0 else self.widths[i]
            w = torch.randn(self.widths[i], self.widths[i + 1], generator=gen, device="cuda") * math.sqrt((2.0 if case["act"] == "relu" and i > 0 else 1.0) / fan_in)
            b = torch.randn(self.widths[i + 1], generator=gen, device="cuda") * 0.1
            self.weights.append(w.cpu().numpy())
            self.biases.append(b.cpu().numpy())
            if last:   # popular items start with a higher score
                popularity = np.empty(items)
                popularity[np.random.default_rng(items).permutation(items)] = np.log(p)
                spread = popularity.std()
                self.biases[-1] += (-3.0 + 0.7 * (popularity - popularity.mean()) / (spread if spread > 0 else 1.0)).astype(np.float32)
        self.start, self.end, self.sparse_index = sparse_rows(rng, rows, items, case["nnz"], p)
        self.nnz = int(self.sparse_index.shape[0])
        self.examples = self.unique_examples = rows
        self.attributes = pkg.ATTR_SPARSE
        self.data_type, self.sparse_data, self.index, self.data_weight = pkg.T_FLOAT, None, None, None
        if case["values"] == "boolean":
            self.attributes |= pkg.ATTR_BOOLEAN
        else:
            dtype = np.dtype(VALUES[case["values"]])
            # ratings: half stars from 0.5 to 5, whole ones from 1 to 5, or bytes (which the layer reads as 256ths)
            stars = rng.integers(1, 11, size=self.nnz)
            self.sparse_data = {"f": stars * 0.5, "i": (stars + 1) // 2, "u": stars * 25}[dtype.kind].astype(dtype)
            self.data_type = pkg.NP_TO_DSX[dtype]
            self.weights[0] *= np.float32(2.0 if dtype.kind == "u" else 0.33)
        if case["weighted"]:
            self.attributes |= pkg.ATTR_WEIGHTED
            self.data_weight = rng.integers(1, 3, rows).astype(np.float32)
        if case["indexed"]:
            self.attributes |= pkg.ATTR_INDEXED
            self.index = rng.permutation(rows).astype(np.uint32)


class State:
    """What a program keeps between calls; gives its device memory back when it is dropped."""

    def __init__(self, case, close, **kept):
        self.case, self.close = case, close
        self.__dict__.update(kept)

    def __del__(self):
        self.close()


def prepare(case, seed):
    pkg = package()
    if case["kind"] in ("serve", "sweep"):
        p = Problem(case, seed)
        net = pkg.host_api.Network(p, max_k=case["k"])
        net.bind_input()
        if case["split"]:
            net.set_split_products(True)
        net.sync()
        p.weights, p.biases, net._keep = None, None, None   # the network has its own copy
        return State(case, net.close, net=net, p=p)
    if case["kind"] == "knn":
        lib = pkg.host_api.load_host_library()
        gen = torch.Generator(device="cuda").manual_seed(seed)
        # embeddings: L2-normalised normal vectors
        items = torch.nn.functional.normalize(torch.randn(case["items"], case["dim"], generator=gen, device="cuda")).cpu().numpy()
        queries = torch.nn.functional.normalize(torch.randn(case["queries"], case["dim"], generator=gen, device="cuda")).cpu().numpy()
        knn = lib.dsstne_knn_create_typed(case["queries"], case["k"], case["storage"].encode())
        if not knn or lib.dsstne_knn_load(knn, items.ctypes.data, case["items"], case["dim"], None) != 0:
            raise RuntimeError(lib.dsstne_last_error().decode())
        return State(case, lambda: lib.dsstne_knn_destroy(knn), lib=lib, knn=knn, queries=queries)
    lib = pkg.init(0)
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    batch, width, k = case["batch"], case["width"], case["k"]
    popularity = torch.randn(width, generator=gen, device="cuda") - 2.0
    scores = torch.sigmoid(torch.randn(batch, width, generator=gen, device="cuda") + popularity)
    kept = dict(scores=scores, keys=torch.empty(batch, k, device="cuda"), values=torch.empty(batch, k, dtype=torch.int32, device="cuda"))
    if case["form"] == "kv":
        kept["payload"] = torch.randint(0, 1 << 31, (batch, width), generator=gen, device="cuda", dtype=torch.int64).to(torch.int32)
    if case["form"] == "filtered":
        start, end, index = sparse_rows(rng, batch, width, min(144, width // 40), item_law(width, 1.0))
        for name, a, dtype in (("start", start, np.int64), ("end", end, np.int64), ("index", index, np.int32)):
            kept[name] = torch.from_numpy(a.astype(dtype)).cuda()
    torch.cuda.synchronize()   # the library's streams are not ordered against torch's
    return State(case, lib.dsx_shutdown, lib=lib, pkg=pkg, **kept)


# --------------------------------------------------------------------------------------------------------------------- work

def serve(s):
    net, p = s.net, s.p
    net.load_sparse(p.start, p.end, p.sparse_data, p.sparse_index)
    net.predict_batch(0)
    net.topk(p.k, filter_dataset="input" if s.case["filtered"] else None)
    return net.get_topk(p.batch)


def sweep(s):
    net, p = s.net, s.p
    results, rows_before = [], 0
    for position in range(0, p.examples, p.batch):
        net.predict_batch(position)
        net.topk(p.k, filter_dataset="input" if s.case["filtered"] else None)
        if position:
            results.append(net.get_topk_previous(rows_before))
        rows_before = min(p.batch, p.examples - position)
    results.append(net.get_topk(rows_before))
    return results


def knn(s):
    queries, k = s.case["queries"], s.case["k"]
    scores, indexes = np.empty((queries, k), np.float32), np.empty((queries, k), np.uint32)
    if s.lib.dsstne_knn_search(s.knn, k, s.queries.ctypes.data, queries, scores.ctypes.data, indexes.ctypes.data) != 0:
        raise RuntimeError(s.lib.dsstne_last_error().decode())
    return scores, indexes


def rank(s):
    c, lib = s.case, s.lib
    common = (s.keys.data_ptr(), s.values.data_ptr(), c["batch"], c["width"], c["k"])
    if c["form"] == "plain":
        rc = lib.dsx_topk(s.scores.data_ptr(), *common)
    elif c["form"] == "kv":
        rc = lib.dsx_topk_kv_u32(s.scores.data_ptr(), s.payload.data_ptr(), *common)
    else:
        rc = lib.dsx_topk_filtered(s.scores.data_ptr(), *common, 0, None, s.start.data_ptr(), s.end.data_ptr(), s.index.data_ptr(), None)
    s.pkg.check(rc)
    return s.keys, s.values


def run(state):
    return {"serve": serve, "sweep": sweep, "knn": knn, "rank": rank}[state.case["kind"]](state)


def work(case):
    """The least one pass can do: inputs, weights and results moved once, every product formed once; scores need not be stored."""
    if case["kind"] == "knn":
        width = 2 if case["storage"] == "fp16" else 4
        return {"bytes": case["items"] * case["dim"] * width + case["queries"] * (4 * case["dim"] + 8 * case["k"]),
                "flops": 2.0 * case["queries"] * case["items"] * case["dim"]}
    if case["kind"] == "rank":
        listed_items = case["batch"] * 144 if case["form"] == "filtered" else 0
        return {"bytes": 4.0 * case["batch"] * case["width"] + 4.0 * listed_items + (8.0 if case["form"] != "kv" else 12.0) * case["batch"] * case["k"], "flops": 0.0}
    nnz = case["rows"] * case["nnz"]
    value = 0 if case["values"] == "boolean" else np.dtype(VALUES[case["values"]]).itemsize
    h, hidden_weights = case["hidden"], (case["depth"] - 1) * case["hidden"] ** 2
    batches = -(-case["rows"] // case["batch"])
    # the weights of the wide layers do not stay in a cache from one batch to the next
    weights = min(nnz, case["items"] * batches) * h + batches * (hidden_weights + h * case["items"])
    return {"bytes": 4.0 * weights + nnz * (4 + value) + case["rows"] * (16 + 8 * case["k"]),
            "flops": 2.0 * nnz * h + 2.0 * case["rows"] * (hidden_weights + h * case["items"])}


def tolerance(case):
    """32-bit sums in another order.  The listed networks and searches compared with themselves with every product formed from
    bf16 pieces (the split-products mode, other roundings and another order of every sum) differ by at most 2.3e-7 (norm) and
    1.3e-6 (single score), and 2.4e-4 of the indexes change places because their scores are that close; deeper drawn networks
    get some room.  A score matrix that is given has one right answer."""
    if case["kind"] == "rank":
        return "exact"
    return {"rel": 2e-6, "max": 1e-5, "differ": 0.001}
