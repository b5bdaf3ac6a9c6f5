"""The work a user of this library has it do, as timed cases over the public entry points: graph search (both
traversal policies, both metrics, one query to a full batch, host and device buffers, with and without tombstones,
beams in LDS and beyond), exact k-nearest neighbours, and graph construction.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a program holds before the call
(the index resident in device memory, its graph, the queries), run() is one call, work() what it cannot do without.
"""
import math

import numpy as np
import torch

from coral_amd import capi

METRICS = {"l2": capi.L2, "ip": capi.IP}
POLICIES = {"rounds": capi.POLICY_ROUNDS, "best_first": capi.POLICY_BEST_FIRST}
R = 32  # row width of every graph (the reference's MAX_DEGREE)
NEIGHBOURS = 100  # base points per auxiliary query in a construction (config.json "k")


def listed():
    return [
        # one user waiting for one answer: latency and launches are all there is
        dict(name="search_one_query", kind="search", entry="host", policy="rounds", metric="l2", n=100000, dim=128,
             graph="exact", aux=0, Q=1, k=10, L=64, deleted=False),
        # a serving loop with small batches through the entry point that allocates nothing and does not wait
        dict(name="search_serving_batch", kind="search", entry="noalloc", policy="rounds", metric="l2", n=200000,
             dim=200, graph="built", aux=20000, Q=64, k=10, L=128, deleted=False),
        # a small best-first batch from host buffers on short odd-sized rows
        dict(name="search_small_best_first", kind="search", entry="host", policy="best_first", metric="ip", n=50001,
             dim=96, graph="exact", aux=0, Q=97, k=10, L=100, deleted=False),
        # the CPU-runnable configuration: 100k x 128, exact 32-NN graph, a thousand queries
        dict(name="search_100k_batch", kind="search", entry="device", policy="rounds", metric="l2", n=100000, dim=128,
             graph="exact", aux=0, Q=1000, k=10, L=64, deleted=False),
        # the headline configuration at its own beam capacity
        dict(name="search_1m_batch", kind="search", entry="device", policy="rounds", metric="l2", n=1000000, dim=200,
             graph="built", aux=50000, Q=10000, k=100, L=512, deleted=False),
        # the CPU path's traversal, a ragged batch
        dict(name="search_best_first_batch", kind="search", entry="device", policy="best_first", metric="l2",
             n=250000, dim=200, graph="built", aux=25000, Q=4999, k=100, L=512, deleted=False),
        # high recall: a beam longer than LDS holds
        dict(name="search_long_beam", kind="search", entry="host", policy="rounds", metric="l2", n=250000, dim=200,
             graph="built", aux=25000, Q=600, k=100, L=4096, deleted=False),
        # image/text embeddings: inner product on unit rows of 512 floats, a tenth of the base deleted
        dict(name="search_ip_deleted", kind="search", entry="device", policy="rounds", metric="ip", n=200000, dim=512,
             graph="built", aux=20000, Q=2000, k=100, L=256, deleted=True),
        # ground truth of a query set (the comp_gt tool)
        dict(name="knn_ground_truth", kind="knn", entry="host", metric="l2", n=1000000, dim=200, Q=10000, k=100,
             deleted=False),
        # exact answers for a handful of queries on a small ragged base
        dict(name="knn_small", kind="knn", entry="device", metric="ip", n=50003, dim=100, Q=100, k=10, deleted=True),
        # construction of a graph from auxiliary queries with the command line's defaults
        dict(name="build_default", kind="build", metric="l2", n=200000, dim=200, aux=20000, top_hit_num=0),
        # construction as the shipped config.json asks for it: the most-hit nodes are searched for and rewired as well
        dict(name="build_top_hits", kind="build", metric="ip", n=60000, dim=512, aux=6000, top_hit_num=5000000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    metric = rng.choice(["l2", "l2", "ip"])
    dim = 4 * _log_int(rng, 16, 128)
    kind = rng.choice(["search", "search", "knn", "build"])
    if kind == "knn":
        return dict(kind="knn", entry=rng.choice(["host", "device"]), metric=metric,
                    n=_log_int(rng, 20000, 500000), dim=dim, Q=_log_int(rng, 1, 10000),
                    k=rng.choice([1, 10, 32, 100, 200]), deleted=rng.random() < 0.3)
    if kind == "build":
        n = _log_int(rng, 30000, 120000)
        return dict(kind="build", metric=metric, n=n, dim=dim, aux=n // rng.choice([8, 10, 13]),
                    top_hit_num=rng.choice([0, 0, 5000000]))
    n = _log_int(rng, 30000, 300000)
    k = rng.choice([1, 10, 50, 100])
    L = _log_int(rng, max(32, k), 1024)
    graph = "exact" if n <= 100000 else "built"
    return dict(kind="search", entry=rng.choice(["host", "device", "noalloc"]),
                policy=rng.choice(["rounds", "rounds", "best_first"]), metric=metric, n=n, dim=dim, graph=graph,
                aux=n // 10 if graph == "built" else 0, Q=_log_int(rng, 1, 5000), k=k, L=L,
                deleted=rng.random() < 0.25)


def _vectors(case, gen, law, count):
    """Rows of the base ("base") or of the queries' law ("queries", "aux"), on the device.  L2: N(0, I) against
    shifted anisotropic queries; inner product: unit rows against queries in a cone (the modality gap of
    text-to-image retrieval)."""
    dim = case["dim"]
    # the law's own parameters come first, so that queries and auxiliary queries share them
    g = torch.Generator(device="cuda")
    g.manual_seed(gen.initial_seed() // 8)
    shift = torch.randn(dim, generator=g, device="cuda")
    scale = 0.5 + torch.rand(dim, generator=g, device="cuda")
    x = torch.randn(count, dim, generator=gen, device="cuda")
    if case["metric"] == "l2":
        return x if law == "base" else 0.5 * shift + scale * x
    if law != "base":
        x = 1.5 * shift / shift.norm() + 0.6 * x
    return x / x.norm(dim=1, keepdim=True)


def _generator(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 8 + stream)
    return g


def _exact_graph(base, metric):
    """Every vector's R nearest others, by the library's exact search."""
    idx = capi.Index(base, None, None, metric=metric)
    ids, _, _ = idx.bruteforce(base, R + 1, want_dists=False)
    idx.close()
    own = ids == np.arange(base.shape[0], dtype=np.int32)[:, None]
    own[~own.any(1), -1] = True
    return ids[~own].reshape(-1, R)


def prepare(case, seed):
    metric = METRICS[case["metric"]]
    n = case["n"]
    base = _vectors(case, _generator(seed, 0), "base", n).cpu().numpy()
    state = dict(case=case)
    if case["kind"] == "build":
        state["aux"] = _vectors(case, _generator(seed, 2), "aux", case["aux"]).cpu().numpy()
        state["params"] = capi.build_params(top_hit_num=case["top_hit_num"])
        state["index"] = capi.Index(base, None, None, metric=metric)
        torch.cuda.synchronize()
        return state
    queries = _vectors(case, _generator(seed, 1), "queries", case["Q"])
    if case["kind"] == "knn":
        index = capi.Index(base, None, None, metric=metric)
    elif case["graph"] == "exact":
        starts = np.random.RandomState(seed % (1 << 32)).choice(n, 16, replace=False).astype(np.int32)
        index = capi.Index(base, _exact_graph(base, metric), starts, metric=metric)
    else:
        index = capi.Index(base, None, None, metric=metric)
        index.build_graph(_vectors(case, _generator(seed, 2), "aux", case["aux"]).cpu().numpy(), capi.build_params())
        index.build_end()
    if case["deleted"]:
        rs = np.random.RandomState((seed + 1) % (1 << 32))
        index.mark_deleted(rs.choice(n, n // 10, replace=False).astype(np.int32))
    if case["kind"] == "search":
        index.prepare(case["Q"], case["L"], policy=POLICIES[case["policy"]])
    state["index"] = index
    if case["entry"] == "host":
        state["queries"] = queries.cpu().numpy()
    else:
        state["queries"] = queries
        state["ids"] = torch.empty((case["Q"], case["k"]), dtype=torch.int32, device="cuda")
        state["dists"] = torch.empty((case["Q"], case["k"]), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    return state


def run(state):
    case, index = state["case"], state["index"]
    if case["kind"] == "build":
        index.build_graph(state["aux"], state["params"])
        nbrs, dists, deg, starts = index.get_graph(with_build_state=True)
        index.build_end()
        return dict(nbrs=nbrs, dists=dists, deg=deg, starts=starts)
    Q, k, deleted, queries = case["Q"], case["k"], case["deleted"], state["queries"]
    if case["kind"] == "knn":
        if case["entry"] == "host":
            ids, dists, _ = index.bruteforce(queries, k, have_delete=deleted)
            return ids, dists
        index.bruteforce_device(queries.data_ptr(), state["ids"].data_ptr(), state["dists"].data_ptr(), Q, k,
                                have_delete=deleted)
        return state["ids"], state["dists"]
    policy, L = POLICIES[case["policy"]], case["L"]
    if case["entry"] == "host":
        ids, dists, _ = index.search(queries, k, L, policy=policy, have_delete=deleted)
        return ids, dists
    if case["entry"] == "device":
        index.search_device(queries.data_ptr(), state["ids"].data_ptr(), state["dists"].data_ptr(), Q, k,
                            policy=policy, have_delete=deleted)
    else:
        index.search_device_noalloc(queries.data_ptr(), state["ids"].data_ptr(), state["dists"].data_ptr(), Q, k, L,
                                    policy=policy, have_delete=deleted)
    return state["ids"], state["dists"]


def _evaluations(case):
    """Distance evaluations of one query: first visits per beam entry, as counted on these data laws (a best-first
    search sees about 20 per entry, the rounds of the other policy about 50), at most the whole base."""
    return min(case["n"], (20 if case["policy"] == "best_first" else 50) * case["L"])


def work(case):
    n, dim = case["n"], case["dim"]
    row, graph_row = 4 * dim, 4 * R
    if case["kind"] == "build":
        A = case["aux"]
        # the clusters' exact neighbours and the distances between the members of every cluster; rows, their
        # distances and their degrees written
        flops = 2.0 * A * n * dim + 3.0 * A * (NEIGHBOURS * (NEIGHBOURS - 1) // 2) * dim
        return dict(bytes=float(n * (row + 2 * graph_row + 4) + A * row), flops=flops)
    Q, k = case["Q"], case["k"]
    io = Q * (row + 8 * k)
    if case["kind"] == "knn":
        return dict(bytes=float(n * row + io), flops=2.0 * Q * n * dim)
    # every row of the index that some query needs once: a vector per evaluation, a graph row per beam entry
    evals = _evaluations(case)
    return dict(bytes=float(min(n, Q * evals) * row + min(n, Q * case["L"]) * graph_row + io),
                flops=(2.0 if case["metric"] == "ip" else 3.0) * Q * evals * dim)


def tolerance(case):
    # ids are whole numbers, ties are ordered by (distance, id), and every distance has a summation order that the
    # library states and keeps: results do not depend on how the work was split
    return "exact"
