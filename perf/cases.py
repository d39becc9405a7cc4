"""Performance cases of the BFS framework: what its users run, through the
public Python entry points, over the range of graphs they run it on.

A case names an operation on a seeded synthetic graph:

  search   DeviceGraph.bfs_device: one search, depths left on the device
  parents  the same plus DeviceGraph.parents_device (a BFS tree)
  host     DeviceGraph.bfs: one search with its depths copied to the host
  batch    DeviceGraph.bfs_batch_device: many sources at once, optionally with
           the row checksums that the server returns with every batch
  csr      csr_build_device: edge tuples to CSR

Graphs are R-MAT (skewed degrees, few levels), uniform random tuples (narrow
degrees) and 4-neighbour grids with 2% of the edges deleted (thousands of
levels). Every output is a whole number, so results are compared for
equality and exact() has nothing to add.
"""
import math

import numpy as np
import torch

from enterprise_amd import DeviceGraph, autotune
from enterprise_amd import _lib as L
from enterprise_amd.convert import csr_build_device

LAUNCH = {"stream": L.LAUNCH_STREAM, "graph": L.LAUNCH_GRAPH}
RMAT_ABC = (0.57, 0.19, 0.19)  # Graph500 quadrant probabilities


def listed():
    return [
        # A small interactive query: everything is latency and launches.
        {"name": "search_rmat10", "op": "search", "graph": "rmat", "n": 1 << 10, "ef": 16},
        # The smoke-test graph: a mid-size query with an odd vertex count.
        {"name": "search_rmat16_odd", "op": "search", "graph": "rmat", "n": 65_001, "ef": 16},
        # The headline benchmark: R-MAT 22 under its tuned configuration.
        {"name": "search_rmat22", "op": "search", "graph": "rmat", "n": 1 << 22, "ef": 16, "tuned": True},
        # A graph larger than the benchmark's, under the default configuration.
        {"name": "search_rmat24", "op": "search", "graph": "rmat", "n": 1 << 24, "ef": 16},
        # High diameter (road-like): thousands of small levels.
        {"name": "search_grid4096", "op": "search", "graph": "grid", "width": 4096, "height": 4096},
        # Narrow degrees, no hubs, ragged size.
        {"name": "search_uniform", "op": "search", "graph": "uniform", "n": 3_000_017, "ef": 8},
        # A BFS tree for a Graph500-style result.
        {"name": "parents_rmat20", "op": "parents", "graph": "rmat", "n": 1 << 20, "ef": 16},
        # The drop-in call with its result handed to host code.
        {"name": "host_rmat20", "op": "host", "graph": "rmat", "n": 1 << 20, "ef": 16},
        # One server batch on the smaller served graph, with its checksums.
        {"name": "batch_rmat20_64", "op": "batch", "graph": "rmat", "n": 1 << 20, "ef": 16, "k": 64,
         "roots": "random", "levels": 8, "hash": True},
        # The multi-source benchmark: hubs and low-degree sources together.
        {"name": "batch_rmat23_512", "op": "batch", "graph": "rmat", "n": 1 << 23, "ef": 16, "k": 512,
         "roots": "mixed", "levels": 48, "tuned": True},
        # The grid's 16 sources as one batch: flushes of the level history.
        {"name": "batch_grid2048_16", "op": "batch", "graph": "grid", "width": 2048, "height": 2048, "k": 16,
         "roots": "random", "levels": 250},
        # The symmetric simple CSR of raw benchmark tuples.
        {"name": "csr_rmat22", "op": "csr", "graph": "rmat", "n": 1 << 22, "ef": 16, "flags": L.CSR_SIMPLE},
    ]


def _log_int(rng, lo, hi):
    """An integer spread over [lo, hi] by its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["search", "search", "search", "parents", "host", "batch", "batch", "csr", "csr"])
    graph = rng.choice(["rmat", "rmat", "uniform", "grid"])
    if op == "csr":
        graph = rng.choice(["rmat", "uniform"])
        n = _log_int(rng, 1 << 10, 1 << 22)
        flags = rng.choice([L.CSR_SIMPLE, L.CSR_SIMPLE, L.CSR_REVERSE, L.CSR_REVERSE | L.CSR_SORT, 0])
        return {"op": op, "graph": graph, "n": n, "ef": rng.randint(1, 16), "flags": flags}
    case = {"op": op, "graph": graph}
    k = _log_int(rng, 2, 512) if op == "batch" else 1
    top = min(1 << 23, (1 << 30) // k) if op == "batch" else 1 << 23
    if graph == "grid":
        # Smaller than the listed grids: levels, not vertices, set their cost.
        cells = _log_int(rng, 1 << 10, min(top, 1 << 22 if k == 1 else 1 << 20))
        width = max(2, int(math.sqrt(cells) * rng.uniform(0.5, 2.0)))
        case.update(width=width, height=max(2, cells // width))
    else:
        case.update(n=_log_int(rng, 1 << 9, top), ef=rng.randint(4, 24))
    if op == "batch":
        case.update(k=k, roots="random" if graph != "rmat" else rng.choice(["random", "mixed"]),
                    levels=rng.choice([8, 32, 48]), hash=rng.random() < 0.5)
    else:
        case.update(tuned=graph == "rmat" and rng.random() < 0.5, launch=rng.choice(["stream", "stream", "graph"]))
    return case


# -- inputs -------------------------------------------------------------------
def _tuples(case, gen):
    """(n, src, dst): the case's raw edge tuples on the GPU."""
    dev = gen.device
    if case["graph"] == "grid":
        w, h = case["width"], case["height"]
        ids = torch.arange(w * h, dtype=torch.int32, device=dev).view(h, w)
        src = torch.cat([ids[:, :-1].reshape(-1), ids[:-1].reshape(-1)])
        dst = torch.cat([ids[:, 1:].reshape(-1), ids[1:].reshape(-1)])
        keep = torch.rand(src.numel(), generator=gen, device=dev) >= 0.02
        return w * h, src[keep], dst[keep]
    n, ne = case["n"], case["n"] * case["ef"]
    if case["graph"] == "uniform":
        ends = torch.randint(0, n, (2, ne), generator=gen, device=dev, dtype=torch.int32)
        return n, ends[0].contiguous(), ends[1].contiguous()
    scale = max(1, (n - 1).bit_length())
    a, b, c = RMAT_ABC
    label = torch.randperm(n, generator=gen, device=dev).to(torch.int32)
    src = torch.empty(ne, dtype=torch.int32, device=dev)
    dst = torch.empty_like(src)
    step = 1 << 25
    for i in range(0, ne, step):
        size = min(step, ne - i)
        u = torch.zeros(size, dtype=torch.int64, device=dev)
        v = torch.zeros_like(u)
        for _ in range(scale):
            r = torch.rand(size, generator=gen, device=dev)
            down, right = r >= a + b, ((r >= a) & (r < a + b)) | (r >= a + b + c)
            u.mul_(2).add_(down)
            v.mul_(2).add_(right)
        # Vertex counts that are no power of two scale the recursion's ids.
        src[i:i + size] = label[(u * n) >> scale]
        dst[i:i + size] = label[(v * n) >> scale]
    return n, src, dst


def _degrees(n, src, dst):
    proper = src != dst
    return torch.bincount(src[proper], minlength=n) + torch.bincount(dst[proper], minlength=n)


def _pick(pool, k, gen):
    """k entries of pool: distinct ones where it holds enough."""
    if pool.numel() >= k:
        return pool[torch.randperm(pool.numel(), generator=gen, device=gen.device)[:k]]
    return pool[torch.randint(0, pool.numel(), (k,), generator=gen, device=gen.device)]


def _roots(case, n, src, dst, gen):
    k = case.get("k", 1)
    deg = _degrees(n, src, dst)
    if case.get("roots") == "mixed":  # half from the top 1% by degree, half of degree 1 to 4
        low = torch.nonzero((deg >= 1) & (deg <= 4)).view(-1)
        if low.numel():
            hubs = torch.topk(deg, max(1, n // 100)).indices
            hubs = hubs[deg[hubs] > 0]
            return torch.cat([_pick(hubs, k - k // 2, gen), _pick(low, k // 2, gen)])
    return _pick(torch.nonzero(deg > 0).view(-1), k, gen)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    n, src, dst = _tuples(case, gen)
    state = {"case": case, "n": n}
    if case["op"] == "csr":
        ne = src.numel()
        cap = ne * (2 if case["flags"] & L.CSR_REVERSE else 1)
        state.update(src=src, dst=dst, ne=ne, cap=cap, beg=torch.empty(n + 1, dtype=torch.int64, device="cuda"),
                     adj=torch.zeros(cap, dtype=torch.int32, device="cuda"))
        return state
    roots = _roots(case, n, src, dst, gen).to(torch.int32).cpu().numpy()
    graph = DeviceGraph.from_edges(n, src.cpu().numpy(), dst.cpu().numpy())
    if case.get("tuned"):
        name = "rmat23_batch" if case["op"] == "batch" else "rmat22"
        tuned = autotune.load(name)
        graph.configure(**{k: v for k, v in tuned.items() if case["op"] != "batch" or k in autotune.BATCH_SPACE})
    if case.get("launch"):
        graph.configure(launch=LAUNCH[case["launch"]])
    state.update(graph=graph, roots=roots, root=int(roots[0]))
    if case["op"] == "batch":
        graph.batch_reserve(case["k"], case["levels"])
        state["depths"] = torch.empty((case["k"], n), dtype=torch.int32, device="cuda")
    elif case["op"] != "host":
        state["depth"] = torch.empty(n, dtype=torch.int32, device="cuda")
        if case["op"] == "parents":
            state["parent"] = torch.empty_like(state["depth"])
    return state


# -- one pass -----------------------------------------------------------------
def _counts(stats):
    return {k: stats[k] for k in ("levels", "reached_vertices", "reached_edges")}


def run(state):
    case = state["case"]
    if case["op"] == "csr":
        m, _ = csr_build_device(state["n"], state["ne"], state["src"].data_ptr(), state["dst"].data_ptr(),
                                case["flags"], state["beg"].data_ptr(), state["adj"].data_ptr(), state["cap"])
        # The whole buffer: entries past m keep what prepare() put there.
        return {"m": m, "beg": state["beg"], "adj": state["adj"]}
    graph = state["graph"]
    if case["op"] == "batch":
        stats = graph.bfs_batch_device(state["roots"], state["depths"].data_ptr())
        out = {"depths": state["depths"], **_counts(stats)}
        if case.get("hash"):
            out["hash"] = graph.row_hash(state["depths"].data_ptr(), case["k"], state["n"]).view(np.int64)
        return out
    if case["op"] == "host":
        depth, stats = graph.bfs(state["root"])
        return {"depth": depth, **_counts(stats)}
    stats = graph.bfs_device(state["root"], state["depth"].data_ptr())
    out = {"depth": state["depth"], **_counts(stats)}
    if case["op"] == "parents":
        graph.parents_device(state["root"], state["depth"].data_ptr(), state["parent"].data_ptr())
        out["parent"] = state["parent"]
    return out


def work(case):
    """Bytes of the inputs and outputs, each once: the CSR (about: repeated
    tuples are merged) and the depth, parent and CSR arrays written."""
    if case["graph"] == "grid":
        n = case["width"] * case["height"]
        ne = 2 * n
    else:
        n, ne = case["n"], case["n"] * case["ef"]
    m = 2 * ne
    if case["op"] == "csr":
        m = ne * (2 if case["flags"] & L.CSR_REVERSE else 1)
        return {"bytes": 8 * ne + 4 * m + 8 * (n + 1), "flops": 0}
    rows = case.get("k", 1) + (1 if case["op"] == "parents" else 0)
    return {"bytes": 8 * (n + 1) + 4 * m + 4 * n * rows, "flops": 0}


def exact(case, seed):
    """Depths, parents, checksums and CSR arrays are whole numbers."""
    return None
