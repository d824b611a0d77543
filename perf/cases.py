"""The work that is timed: what a program that trains node embeddings on random
walks asks of this package, from the edge list to the skip-gram windows.

Every case goes through the package's Python entry points with the arguments
such a program gives, and with their default checks (a walk call waits for its
status word, a graph build for its entry count).

Kinds of case:
  uniform   random_walk: uniform walks over a CSR graph
  node2vec  rejection_sampling: second-order walks (p, q)
  csr       to_csr: an edge list turned into the CSR that the walks read
  windows   context_windows and negative_windows of finished walks

Graphs: "cora" is a preferential-attachment graph with about 2 pairs a node
(the citation graphs of the small examples), "rmat" the skewed R-MAT graphs of
the benchmark, "hubs" a preferential-attachment graph with hub nodes added.
"""
import math

import torch

import mlx_cluster_amd as mlx_cluster
from mlx_cluster_amd import synth


def listed():
    return [
        # The reference tests' own call: 2,000 walks of 5 steps on a graph of
        # Cora's size.  Launches and the wait for the status word count here.
        {"name": "uniform cora", "kind": "uniform", "graph": "cora", "nodes": 2708, "edges": 5278,
         "symmetrize": True, "walks": 2000, "starts": "first", "length": 5, "seeded": False,
         "int32": False, "return_edges": False},
        # One mini-batch of a training loop on a large graph: 130 shuffled
        # nodes, 10 walks each, uniforms drawn in the kernel, compact output
        # with the edge ids (to look up edge features).
        {"name": "uniform batch", "kind": "uniform", "graph": "rmat", "nodes": 1 << 20,
         "edges": 1 << 24, "symmetrize": False, "walks": 1300, "starts": "random", "length": 37,
         "seeded": True, "int32": True, "return_edges": True},
        # An epoch's walks over every node of a mid-size graph, uniforms given:
        # the headline workload of the benchmark.
        {"name": "uniform epoch", "kind": "uniform", "graph": "rmat", "nodes": 1 << 20,
         "edges": 1 << 24, "symmetrize": False, "walks": 10 << 20, "starts": "all", "length": 80,
         "seeded": False, "int32": False, "return_edges": False},
        # One walk from every node of a graph far larger than the caches.
        {"name": "uniform large graph", "kind": "uniform", "graph": "rmat", "nodes": 1 << 24,
         "edges": 1 << 28, "symmetrize": False, "walks": 1 << 24, "starts": "all", "length": 20,
         "seeded": False, "int32": False, "return_edges": False},
        # The reference's rejection-sampling test: p = 1, q = 3.
        {"name": "node2vec cora", "kind": "node2vec", "graph": "cora", "nodes": 2708,
         "edges": 5278, "symmetrize": True, "walks": 2000, "starts": "first", "length": 5,
         "p": 1.0, "q": 3.0, "rule": "ref_chain", "symmetric": False, "int32": False,
         "return_edges": False},
        # A mini-batch of node2vec training on a large undirected graph.
        {"name": "node2vec batch", "kind": "node2vec", "graph": "rmat", "nodes": 1 << 20,
         "edges": 1 << 24, "symmetrize": True, "walks": 1300, "starts": "random", "length": 40,
         "p": 0.5, "q": 2.0, "rule": "ref_chain", "symmetric": False, "int32": False,
         "return_edges": False},
        # An epoch's node2vec walks over every node of the same graph.
        {"name": "node2vec epoch", "kind": "node2vec", "graph": "rmat", "nodes": 1 << 20,
         "edges": 1 << 24, "symmetrize": True, "walks": 4 << 20, "starts": "all", "length": 40,
         "p": 0.5, "q": 2.0, "rule": "ref_chain", "symmetric": False, "int32": False,
         "return_edges": False},
        # The analytic rule at p = 4, q = 0.25 on a graph with hubs of 500,000
        # neighbours, where many candidates are rejected; node count not a
        # power of two.
        {"name": "node2vec hubs", "kind": "node2vec", "graph": "hubs", "nodes": 4_000_000,
         "edges": 80_000_000, "symmetrize": True, "walks": 8_000_000, "starts": "all",
         "length": 30, "p": 4.0, "q": 0.25, "rule": "node2vec", "symmetric": False,
         "int32": False, "return_edges": False},
        # The CSR of a small data set's edge list, duplicates kept, as the
        # reference's tests build theirs: launches count.
        {"name": "csr cora", "kind": "csr", "graph": "cora", "nodes": 2708, "edges": 10556,
         "distinct": 10556, "symmetrize": False, "dedup": False},
        # An undirected graph from one list of pairs: reversed pairs added,
        # duplicates merged; sizes that are no powers of two.
        {"name": "csr undirected", "kind": "csr", "graph": "rmat", "nodes": 1_000_003,
         "edges": 15_000_001, "distinct": 14_000_000, "symmetrize": True, "dedup": True},
        # The CSR of the large graph.
        {"name": "csr large graph", "kind": "csr", "graph": "rmat", "nodes": 1 << 24,
         "edges": 1 << 28, "distinct": 262_000_000, "symmetrize": False, "dedup": True},
        # Skip-gram windows of a large batch of walks, with as many negative
        # ones: walk length 20, context 10.
        {"name": "windows", "kind": "windows", "nodes": 1 << 20, "walks": 1_000_003,
         "length": 20, "context": 10, "int32": False},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["uniform", "uniform", "node2vec", "node2vec", "csr", "csr", "windows"])
    if kind == "windows":
        context = rng.randint(2, 16)
        return {"kind": kind, "nodes": _log_uniform(rng, 1 << 11, 1 << 24),
                "walks": _log_uniform(rng, 100, 1_000_000), "length": rng.randint(context, 30),
                "context": context, "int32": rng.random() < 0.3}
    if kind == "csr":
        nodes = _log_uniform(rng, 1 << 10, 1 << 24)
        symmetrize = rng.random() < 0.5
        edges = _log_uniform(rng, 2 * nodes, 16 * nodes) // (2 if symmetrize else 1)
        return {"kind": kind, "graph": "rmat", "nodes": nodes, "edges": edges,
                "distinct": edges * 7 // 10, "symmetrize": symmetrize, "dedup": rng.random() < 0.7}
    nodes = _log_uniform(rng, 1 << 11, 1 << (24 if kind == "uniform" else 21))
    edges = _log_uniform(rng, 4 * nodes, 16 * nodes)
    length = rng.randint(5, 80 if kind == "uniform" else 40)
    most = (300_000_000 if kind == "uniform" else 80_000_000) // length
    case = {"kind": kind, "graph": "rmat", "nodes": nodes, "edges": edges,
            "symmetrize": kind == "node2vec" or rng.random() < 0.3,
            "walks": _log_uniform(rng, 200, min(most, 10 * nodes)), "length": length,
            "starts": rng.choice(["random", "all"]), "int32": rng.random() < 0.3,
            "return_edges": rng.random() < 0.2}
    if kind == "uniform":
        case["seeded"] = rng.random() < 0.4
    else:
        case["p"] = rng.choice([0.25, 0.5, 1.0, 4.0])
        case["q"] = rng.choice([0.25, 0.5, 2.0, 3.0])
        case["rule"] = rng.choice(["ref_chain", "node2vec"])
        case["symmetric"] = rng.random() < 0.3
    return case


def _rmat_pairs(case, seed):
    V, E = case["nodes"], case["edges"]
    row, col = synth.rmat_edges(max(1, (V - 1).bit_length()), E, seed=seed, device="cuda")
    return row.remainder_(V), col.remainder_(V)


def _edge_list(case, seed):
    """R-MAT pairs in random order, exactly case["distinct"] of them different
    (as undirected pairs, no loops, when the build symmetrizes), the others
    repeats, so that every seed's CSR has the same number of entries."""
    V, E, K = case["nodes"], case["edges"], case["distinct"]
    row, col = _rmat_pairs(case, seed)
    if case["symmetrize"]:
        keys = (torch.minimum(row, col) * V + torch.maximum(row, col))[row != col]
    else:
        keys = row * V + col
    del row, col
    keys = torch.unique(keys)
    if keys.numel() < K:
        raise ValueError(f"{keys.numel()} distinct pairs, {K} wanted")
    g = torch.Generator(device="cuda").manual_seed(seed)
    keys = keys[torch.randperm(keys.numel(), generator=g, device="cuda")[:K]]
    keys = torch.cat([keys, keys[torch.randint(0, K, (E - K,), generator=g, device="cuda")]])
    keys = keys[torch.randperm(E, generator=g, device="cuda")]
    return torch.stack([keys // V, keys % V])


def _graph(case, seed):
    V, E = case["nodes"], case["edges"]
    if case["graph"] == "cora":
        rowptr, col = synth.cora_like(seed, V, E)
        return torch.from_numpy(rowptr).cuda(), torch.from_numpy(col).cuda()
    if case["graph"] == "hubs":
        return synth.ba_hub_csr(V, E // V, 64, V // 8, seed=seed, device="cuda")
    return mlx_cluster.to_csr(torch.stack(_rmat_pairs(case, seed)), V,
                              symmetrize=case["symmetrize"], dedup=True)


def prepare(case, seed):
    kind, V = case["kind"], case["nodes"]
    if kind == "csr":
        if case["graph"] == "cora":
            rowptr, col = synth.cora_like(seed, V, case["edges"] // 2)
            degree = torch.from_numpy(rowptr).diff()
            pairs = torch.stack([torch.arange(V).repeat_interleave(degree), torch.from_numpy(col)])
            order = torch.randperm(pairs.shape[1], generator=torch.Generator().manual_seed(seed))
            return {"case": case, "edge_index": pairs[:, order].cuda()}
        return {"case": case, "edge_index": _edge_list(case, seed)}
    g = torch.Generator(device="cuda").manual_seed(seed)
    N, L = case["walks"], case["length"]
    if kind == "windows":
        dtype = torch.int32 if case["int32"] else torch.int64
        walks = torch.randint(0, V, (N, L + 1), generator=g, device="cuda", dtype=dtype)
        return {"case": case, "seed": seed, "walks": walks, "start": walks[:, 0].long()}
    rowptr, col = _graph(case, seed)
    if case["starts"] == "random":  # a shuffled loader's nodes, ten walks each
        start = torch.randint(0, V, (-(-N // 10),), generator=g, device="cuda").repeat(10)[:N]
    else:  # the nodes in order, over and over
        start = torch.arange(N, device="cuda") % V
    state = {"case": case, "seed": seed, "rowptr": rowptr, "col": col, "start": start}
    if kind == "uniform" and not case["seeded"]:
        state["rand"] = torch.rand(N, L, generator=g, device="cuda")
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "csr":
        return mlx_cluster.to_csr(state["edge_index"], case["nodes"],
                                  symmetrize=case["symmetrize"], dedup=case["dedup"])
    if kind == "windows":
        L, C = case["length"], case["context"]
        return (mlx_cluster.context_windows(state["walks"], C),
                mlx_cluster.negative_windows(state["start"], L, C, case["nodes"],
                                             seed=state["seed"],
                                             out_dtype=state["walks"].dtype))
    graph = state["rowptr"], state["col"], state["start"]
    options = {"return_edges": case["return_edges"],
               "out_dtype": torch.int32 if case["int32"] else torch.int64}
    if kind == "uniform":
        if case["seeded"]:
            return mlx_cluster.random_walk(*graph, None, case["length"], seed=state["seed"],
                                           **options)
        return mlx_cluster.random_walk(*graph, state["rand"], case["length"], **options)
    return mlx_cluster.rejection_sampling(*graph, case["length"], case["p"], case["q"],
                                          seed=state["seed"], rule=case["rule"],
                                          symmetric=case["symmetric"], **options)


def work(case):
    """Each input read once, or as much of it as the walks' steps can touch,
    and each output written once."""
    kind, V = case["kind"], case["nodes"]
    if kind == "windows":
        N, L, C = case["walks"], case["length"], case["context"]
        size = 4 if case["int32"] else 8
        windows = N * (L + 2 - C)
        return {"bytes": N * (L + 1) * size + N * 8 + 2 * windows * C * size}
    if kind == "csr":
        entries = case["distinct" if case["dedup"] else "edges"]
        entries *= 2 if case["symmetrize"] else 1
        return {"bytes": 16 * case["edges"] + 8 * (V + 1) + 8 * entries}
    entries = case["edges"] * (2 if case["symmetrize"] else 1)
    N, L = case["walks"], case["length"]
    size = 4 if case["int32"] else 8
    written = N * (L + 1) * size + (N * L * size if case["return_edges"] else 0)
    if kind == "uniform":
        # a walk reads the rows it leaves (two bounds) and the entry it takes
        graph = min(8 * (V + 1), 16 * N * L) + min(8 * entries, 8 * N * L)
        rand = 0 if case["seeded"] else 4 * N * L
        return {"bytes": graph + 8 * N + rand + written}
    # a node2vec call also checks the whole graph
    return {"bytes": 8 * (V + 1) + 8 * entries + 8 * N + written}


def tolerance(case):
    """Node and edge ids: the same inputs have one right answer."""
    return "exact"


def exact(case, seed):
    """The outputs are whole numbers, which are compared as they are."""
    return None
