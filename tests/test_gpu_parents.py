"""GPU parent output: for every search the parents form a BFS tree that
passes the Graph500 parent checks of the oracle (parent[root] = root, each
parent a neighbour one level closer, -1 for unreached vertices), with depths
bit-exact against the oracle; depths that are not a BFS from the given root
are rejected."""
import sys

import numpy as np
import pytest

import graphs
from enterprise_amd import DeviceGraph, HostGraph
from enterprise_amd import _lib as L

pytestmark = pytest.mark.gpu


def _check(oracle, g, dg, root, tag):
    print(f"[gpu] parents {tag} root={root}", flush=True)
    sys.stdout.flush()
    d, p, st = dg.bfs_parents(root)
    assert np.array_equal(d, oracle.bfs(g.beg_pos, g.adj, root)), tag
    rc = oracle.validate_parents(g.beg_pos, g.adj, root, d, p)
    assert rc == 0, (tag, root, rc)
    assert p[root] == root
    assert (p[d < 0] == -1).all()
    return p


@pytest.mark.parametrize("name", list(graphs.CLOSED_FORMS))
def test_parents_closed_forms(oracle, name):
    g, _ = graphs.CLOSED_FORMS[name]()
    with DeviceGraph(g) as dg:
        for r in sorted({0, g.n // 2, g.n - 1}):
            _check(oracle, g, dg, r, name)


@pytest.mark.parametrize("keep_order", [False, True])
def test_parents_rmat16(oracle, keep_order):
    g = HostGraph.rmat(16, 16, seed=16)
    with DeviceGraph(g, keep_order=keep_order) as dg:
        for r in g.pick_roots(6, 31):
            _check(oracle, g, dg, int(r), f"rmat16/keep{keep_order}")
        dg.configure(direction=L.DIR_BOTTOMUP)
        _check(oracle, g, dg, int(g.pick_roots(1, 32)[0]), "rmat16/bu")


def test_parents_star_hub_and_leaf(oracle):
    g, _ = graphs.star(70000)
    with DeviceGraph(g) as dg:
        p = _check(oracle, g, dg, 0, "star/hub")
        assert (p[1:] == 0).all()
        p = _check(oracle, g, dg, 5, "star/leaf")
        assert p[0] == 5 and (np.delete(p, [0, 5]) == 0).all()


def test_parents_reject_foreign_depths():
    g = HostGraph.rmat(12, 8, seed=3)
    a, b = (int(x) for x in g.pick_roots(2, 9))
    with DeviceGraph(g) as dg:
        buf = dg.device_alloc(8 * g.n)
        try:
            dg.bfs_device(a, buf)                     # depths of a search from a
            with pytest.raises(L.EntError) as e:      # ... are no BFS from b
                dg.parents_device(b, buf, buf + 4 * g.n)
            assert e.value.code == L.ENT_EINVAL
            dg.parents_device(a, buf, buf + 4 * g.n)  # and are one from a
        finally:
            dg.device_free(buf)


def _first_parents(beg, adj, depth, root):
    """The first neighbour one level closer of every reached vertex."""
    rows = np.repeat(np.arange(beg.size - 1), np.diff(beg))
    pos = np.where(depth[adj] == depth[rows] - 1, np.arange(adj.size), adj.size)
    first = np.full(beg.size - 1, adj.size, np.int64)
    np.minimum.at(first, rows, pos)
    par = np.full(beg.size - 1, -1, np.int64)
    hit = (first < adj.size) & (depth > 0)
    par[hit] = adj[first[hit]]
    par[root] = root
    return par


@pytest.mark.parametrize("pos", [0, 15, 16, 1039, 1040, 1041, 2063, 2064, 9000, 39997])
def test_parents_long_rows(oracle, pos):
    """Three hubs of 40,000 neighbours whose parent sits at row position pos
    (and again two entries later), at the edges of the lane probe, the
    wavefront's share and the pieces of the long-row kernel."""
    hubs, leaves = 3, 39998
    p1, p2, root = hubs, hubs + 1, hubs + 2
    first_leaf = root + 1
    n = first_leaf + hubs * leaves
    rows = [[] for _ in range(n)]
    for h in range(hubs):
        mine = list(range(first_leaf + h * leaves, first_leaf + (h + 1) * leaves))
        for v in mine:
            rows[v] = [h]
        q = min(pos + h, leaves)
        rows[h] = mine[:q] + [p1] + mine[q:q + 1] + [p2] + mine[q + 1:]
    rows[p1] = rows[p2] = list(range(hubs)) + [root]
    rows[root] = [p1, p2]
    beg = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64)
    adj = np.concatenate([np.array(r, np.int32) for r in rows])
    with DeviceGraph(beg_pos=beg, adj=adj, keep_order=True) as dg:
        for r in (root, first_leaf):
            print(f"[gpu] parents long rows pos={pos} root={r}", flush=True)
            d, p, _ = dg.bfs_parents(r)
            assert np.array_equal(d, oracle.bfs(beg, adj, r))
            assert np.array_equal(p, _first_parents(beg, adj, d, r))
        # A hub without a neighbour one level closer is counted and marked.
        buf = dg.device_alloc(8 * n)
        try:
            dg.bfs_device(root, buf)
            with pytest.raises(L.EntError) as e:
                dg.parents_device(first_leaf, buf, buf + 4 * n)
            assert e.value.code == L.ENT_EINVAL
            dg.parents_device(root, buf, buf + 4 * n)
        finally:
            dg.device_free(buf)
