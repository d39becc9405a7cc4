"""GPU parity of the several-levels-per-launch searches (bfs_deep.hip) on
graphs of low degree and high diameter: depths and counts against the oracle
at the edges of a launch's levels, on graphs with odd cycles (a block can
reach a vertex by the longer way first), at the largest degree of the rule,
and on graphs that spread too fast and fall back; batches of few sources
against single-source rows and the joint search's counts."""
import ctypes as C

import numpy as np
import pytest

import graphs
from enterprise_amd import DeviceGraph, HostGraph
from enterprise_amd import _lib as L

pytestmark = pytest.mark.gpu

LAUNCHES = {"stream": L.LAUNCH_STREAM, "graph": L.LAUNCH_GRAPH}
COUNTS = ("levels", "reached_vertices", "reached_edges", "td_levels")


def _say(msg):
    print(msg, flush=True)


def _random_grid(w, h, diagonals, seed):
    """Grid with 10% of its edges deleted and random diagonals (odd cycles)."""
    rng = np.random.default_rng(seed)
    ids = np.arange(w * h).reshape(h, w)
    e = np.concatenate([np.stack([ids[:, :-1].ravel(), ids[:, 1:].ravel()], 1),
                        np.stack([ids[:-1].ravel(), ids[1:].ravel()], 1)])
    e = e[rng.random(len(e)) > 0.1]
    d = np.stack([ids[:-1, :-1].ravel(), ids[1:, 1:].ravel()], 1)
    return graphs.edges_graph(w * h, np.concatenate([e, d[rng.random(len(d)) < diagonals]]))


def _caterpillar(spine, legs):
    """A path whose inner vertices have `legs` leaves each (degree legs + 2)."""
    e = [(i, i + 1) for i in range(spine - 1)]
    e += [(i, spine + i * legs + j) for i in range(spine) for j in range(legs)]
    return graphs.edges_graph(spine + spine * legs, e)


def _path_then_tree(length, branch, levels):
    """A path into a complete tree of `branch` children per vertex: small
    frontiers first, then ones that outgrow a block's queue in one launch."""
    e, n, last = [(i, i + 1) for i in range(length - 1)], length, [length - 1]
    for _ in range(levels):
        nxt = []
        for v in last:
            for _ in range(branch):
                e.append((v, n))
                nxt.append(n)
                n += 1
        last = nxt
    return graphs.edges_graph(n, e)


CASES = {
    # Paths that end just before, at and after a launch's last level.
    **{f"path{n}": (lambda n=n: graphs.path(n)[0]) for n in (13, 20, 21, 22, 23, 28, 29, 30, 31, 37, 300)},
    "cycle513": lambda: graphs.cycle(513)[0],
    "disjoint": lambda: graphs.disjoint_paths(100, 77)[0],
    "grid200x150": lambda: _random_grid(200, 150, 0.0, 1),
    "diagonals200x150": lambda: _random_grid(200, 150, 0.3, 2),
    "diagonals700x31": lambda: _random_grid(700, 31, 0.05, 3),
    "degree16": lambda: _caterpillar(300, 14),
    "degree17": lambda: _caterpillar(300, 15),  # beyond the rule
    "spreads": lambda: _path_then_tree(40, 15, 4),
    "bintree11": lambda: graphs.binary_tree(11)[0],
}


@pytest.mark.parametrize("launch", list(LAUNCHES))
@pytest.mark.parametrize("name", list(CASES))
def test_deep_search(oracle, name, launch):
    g = CASES[name]()
    rng = np.random.default_rng(5)
    deg = np.diff(g.beg_pos)
    roots = [int(np.flatnonzero(deg)[0])] + [int(r) for r in rng.choice(np.flatnonzero(deg), 4)]
    with DeviceGraph(g) as dg:
        for direction in (L.DIR_AUTO, L.DIR_TOPDOWN, L.DIR_AUTO):
            dg.configure(launch=LAUNCHES[launch], direction=direction)
            for r in roots:
                want = oracle.bfs(g.beg_pos, g.adj, r)
                _say(f"[gpu] deep {name} {launch} dir={direction} root={r}")
                got, st = dg.bfs(r)
                assert np.array_equal(got, want), (name, r)
                edges, verts = oracle.report(g.beg_pos, want)
                assert (st["reached_edges"], st["reached_vertices"]) == (edges, verts), st
                assert st["levels"] == int(want.max()) + 1, st
                if direction == L.DIR_TOPDOWN:
                    assert st["td_levels"] == st["levels"], st
        if name == "path300":  # the form did run: fewer launches than levels
            _, st = dg.bfs(0)
            assert st["levels"] == 300 and st["phases"] < 100, st


def _refused_then_tail(legs, tail):
    """More vertices than one block searches: a binary tree whose frontiers
    double until level 13 (a hand-over there is refused), a path of `tail`
    vertices at its last leaf, `legs` leaves at each of them."""
    levels = 14
    leaf = (1 << levels) - 2
    e = [(v, (v - 1) // 2) for v in range(1, leaf + 1)]
    spine = [leaf] + list(range(leaf + 1, leaf + 1 + tail))
    e += list(zip(spine[:-1], spine[1:]))
    n = spine[-1] + 1
    for v in spine[1:]:
        e += [(v, n + j) for j in range(legs)]
        n += legs
    return graphs.edges_graph(max(n, (1 << 14) + 1), e)


@pytest.mark.parametrize("launch", list(LAUNCHES))
@pytest.mark.parametrize("legs", [0, 5, 14])
def test_deep_refused_hand_over(oracle, legs, launch):
    """Hand-overs refused early in a search (its frontiers grow), then one that
    is taken, with a tail of several launches behind it: depths and counts on
    the same handle again and again, and from roots inside the tail. One case
    per row form (padded rows of 4 and 8 entries, CSR)."""
    for tail in (30, 60, 700):
        g = _refused_then_tail(legs, tail)
        deg = np.diff(g.beg_pos)
        assert deg.max() == max(3, legs + 2)
        with DeviceGraph(g) as dg:
            for direction in (L.DIR_TOPDOWN, L.DIR_AUTO):
                dg.configure(launch=LAUNCHES[launch], direction=direction)
                for r in (0, 1, 0, (1 << 14) - 2 + tail // 2, 0):
                    want = oracle.bfs(g.beg_pos, g.adj, r)
                    _say(f"[gpu] deep refused hand-over legs={legs} tail={tail} {launch} dir={direction} root={r}")
                    got, st = dg.bfs(r)
                    assert np.array_equal(got, want), (r, np.flatnonzero(got != want)[:8])
                    edges, verts = oracle.report(g.beg_pos, want)
                    assert (st["reached_edges"], st["reached_vertices"]) == (edges, verts), st
                    assert st["levels"] == int(want.max()) + 1, st


def test_deep_directed_topdown(oracle):
    """Forced top-down on a directed ring with chords and vertices that have
    in-edges only."""
    n = 900
    beg, adj = [0], []
    for v in range(n):
        row = sorted({(v + 1) % 600, 600 + v % 300} | ({(v + 7) % 600} if v % 3 == 0 else set())) if v < 600 else []
        adj += row
        beg.append(len(adj))
    g = HostGraph.from_arrays(np.array(beg, np.int64), np.array(adj, np.int32))
    with DeviceGraph(g, keep_order=True) as dg:
        dg.configure(direction=L.DIR_TOPDOWN)
        for r in (0, 1, 599):
            _say(f"[gpu] deep directed root={r}")
            got, st = dg.bfs(r)
            assert np.array_equal(got, oracle.bfs(g.beg_pos, g.adj, r))
            assert st["phases"] < st["levels"]


@pytest.mark.parametrize("k", [1, 2, 15, 16, 17, 32, 33, 64, 65, 200])
def test_deep_batch(oracle, k):
    """Batches on a 300 x 250 grid with odd cycles: every row equals the
    oracle's, and the counts equal the joint search's on the same roots.
    Unaligned output too."""
    g = _random_grid(300, 250, 0.1, 7)
    roots = g.pick_roots(k, 11)
    if k > 2:
        roots[1] = roots[0]  # a repeated root
    want = np.stack([oracle.bfs(g.beg_pos, g.adj, int(r)) for r in roots])
    with DeviceGraph(g) as dg:
        dg.batch_reserve(k, 40)
        _say(f"[gpu] deep batch k={k}")
        out, st = dg.bfs_batch(roots)
        assert np.array_equal(out, want)
        dg.configure(batch_fused=0)  # the joint search, one level at a time
        joint, sj = dg.bfs_batch(roots)
        assert np.array_equal(joint, want)
        for key in ("levels", "reached_vertices", "reached_edges", "alg_bytes", "words", "k", "flushes"):
            assert st[key] == sj[key], (key, st, sj)
        assert 8 * st["phases"] < sj["phases"]
        dg.configure(batch_fused=8)
        single, _ = dg.bfs(int(roots[0]))  # one mirror serves both forms
        assert np.array_equal(single, want[0])
        dev = dg.device_alloc(4 * k * g.n + 4)
        try:
            dg.bfs_batch_device(roots, dev + 4)
            assert np.array_equal(dg.copy_depth(dev + 4, k * g.n).reshape(k, g.n), want)
        finally:
            dg.device_free(dev)


def test_deep_batch_spreading_graph(oracle):
    """A tree of 15 children per vertex: the frontiers outgrow the queues and
    the batch runs as a joint search, the second time from the start."""
    g = _path_then_tree(12000, 15, 4)
    assert g.n >= 1 << 16
    with DeviceGraph(g) as dg:
        for roots in ([11990, 11999], [5, 12040]):
            _say(f"[gpu] deep batch, spreading graph, roots {roots}")
            out, st = dg.bfs_batch(np.array(roots, np.int32))
            for i, r in enumerate(roots):
                assert np.array_equal(out[i], oracle.bfs(g.beg_pos, g.adj, r))


def _limit(dg, nbytes):
    f = L.lib().ent_internal_limit_device_bytes
    f.argtypes, f.restype = [C.c_void_p, C.c_int64], C.c_int
    assert f(dg.handle, nbytes) == L.ENT_OK


def test_deep_search_without_room(oracle):
    """A handle whose tables for several levels per launch cannot be had
    searches in the ordinary form."""
    g = _random_grid(200, 150, 0.1, 4)
    roots = [int(r) for r in g.pick_roots(3, 2)]
    with DeviceGraph(g) as dg, DeviceGraph(share=dg) as roomy:
        _limit(dg, roomy.info()["device_bytes"] - 64)
        with DeviceGraph(share=dg) as tight:
            for launch in LAUNCHES.values():
                for h in (tight, roomy):
                    h.configure(launch=launch)
                for r in roots:
                    _say(f"[gpu] deep search without room, launch {launch} root={r}")
                    want = oracle.bfs(g.beg_pos, g.adj, r)
                    got, st = tight.bfs(r)
                    assert np.array_equal(got, want)
                    got, sr = roomy.bfs(r)
                    assert np.array_equal(got, want)
                    assert 2 * sr["phases"] < sr["levels"] < st["phases"]
                    for key in COUNTS[:3]:
                        assert st[key] == sr[key], (key, st, sr)


def test_deep_batch_without_room(oracle):
    """A batch workspace that has room for the joint search alone serves the
    batch as one, and the same handle side by side once there is room."""
    g = _random_grid(300, 250, 0.1, 7)
    k = 70
    roots = g.pick_roots(k, 11)
    want = np.stack([oracle.bfs(g.beg_pos, g.adj, int(r)) for r in roots])
    with DeviceGraph(g) as dg:
        # One byte less than all of it, which leaves room for the library's own
        # rows of bfs_batch.
        need = L.lib().ent_batch_workspace_bytes(dg.handle, k, 40)
        _limit(dg, dg.info()["device_bytes"] + need - 1)
        dg.batch_reserve(k, 40)
        _say("[gpu] deep batch without room")
        out, st = dg.bfs_batch(roots)
        assert np.array_equal(out, want)
        assert st["phases"] >= st["levels"]
        dg.batch_release()
        _limit(dg, 0)
        before = dg.info()["device_bytes"]
        dg.batch_reserve(k, 40)
        assert dg.info()["device_bytes"] - before == need
        side, ss = dg.bfs_batch(roots)
        assert np.array_equal(side, want)
        assert 8 * ss["phases"] < st["phases"]
        for key in ("levels", "reached_vertices", "reached_edges", "alg_bytes", "words", "k", "flushes"):
            assert st[key] == ss[key], (key, st, ss)
        # A smaller batch, then one as large as the workspace takes.
        for m in (3, 128):
            r = g.pick_roots(m, m)
            out, ss = dg.bfs_batch(r)
            assert np.array_equal(out, np.stack([oracle.bfs(g.beg_pos, g.adj, int(x)) for x in r]))
            assert 8 * ss["phases"] < st["phases"]


def test_deep_spreading_graph_is_known_to_every_handle(oracle):
    """What one handle's first batch (search) finds out about the graph holds
    for the others: their workspaces leave the tables out, and their first
    batch is a joint search."""
    rng = np.random.default_rng(3)
    n = 1 << 15
    e = rng.integers(0, n, (2, n))  # mean degree 2: outgrows a block within ten levels
    g = HostGraph.from_edges(n, e[0], e[1])
    assert 8 < np.diff(g.beg_pos).max() <= 16
    roots = g.pick_roots(40, 3)
    want = np.stack([oracle.bfs(g.beg_pos, g.adj, int(r)) for r in roots])
    with DeviceGraph(g) as dg, DeviceGraph(share=dg) as other:
        before = L.lib().ent_batch_workspace_bytes(other.handle, 40, 32)
        other.batch_reserve(40, 32)
        for h in (dg, dg, other):
            _say("[gpu] deep spreading batch")
            out, st = h.bfs_batch(roots)
            assert np.array_equal(out, want)
            assert st["phases"] >= st["levels"]  # the joint search
        for h in (dg, other):
            assert L.lib().ent_batch_workspace_bytes(h.handle, 40, 32) < before


ABOVE_ONE_BLOCK = (1 << 14) + 1  # vertices; smaller graphs are searched by one block


def _padded(g):
    """g with isolated vertices behind it, so that one block does not take it."""
    n = max(g.n, ABOVE_ONE_BLOCK)
    beg = np.concatenate([g.beg_pos, np.full(n - g.n, g.beg_pos[-1], dtype=np.int64)])
    return HostGraph.from_arrays(beg, np.array(g.adj, dtype=np.int32))


def _agrees(oracle, g, dg, root):
    want = oracle.bfs(g.beg_pos, g.adj, root)
    got, st = dg.bfs(root)
    assert np.array_equal(got, want), (root, np.flatnonzero(got != want)[:8])
    assert (st["reached_edges"], st["reached_vertices"]) == oracle.report(g.beg_pos, want), st
    assert st["levels"] == int(want.max()) + 1, st
    return st


@pytest.mark.parametrize("launch", list(LAUNCHES))
@pytest.mark.parametrize("direction", ["topdown", "auto"])
def test_deep_ends_of_launches(oracle, direction, launch):
    """Paths of every length from 8 to 100 in one graph: searches that end
    before the hand-over and at each level of the first launches behind it."""
    lengths = range(8, 101)
    edges, first = [], []
    n = 0
    for k in lengths:
        first.append(n)
        edges += [(n + i, n + i + 1) for i in range(k - 1)]
        n += k
    g = _padded(graphs.edges_graph(n, edges))
    with DeviceGraph(g) as dg:
        dg.configure(launch=LAUNCHES[launch], direction=L.DIR_TOPDOWN if direction == "topdown" else L.DIR_AUTO)
        for k, v in zip(lengths, first):
            _say(f"[gpu] deep path of {k}, {direction}, {launch}")
            st = _agrees(oracle, g, dg, v)
            _agrees(oracle, g, dg, v + k // 2)
            # Several levels a launch, behind as many launches as the search
            # before it took (at most k / 2 + 2).
            if k >= 64:
                assert 1 < st["phases"] < st["levels"], st


@pytest.mark.parametrize("launch", list(LAUNCHES))
@pytest.mark.parametrize("legs", [0, 2, 3, 6, 7, 14, 15])
def test_deep_row_forms(oracle, legs, launch):
    """Long spines whose vertices have `legs` leaves: both sides of the degrees
    at which rows are padded to 4 and 8 entries, the CSR form up to the largest
    degree, and the degree beyond it."""
    g = _padded(_caterpillar(1200, legs))
    assert np.diff(g.beg_pos).max() == legs + 2
    with DeviceGraph(g) as dg:
        for direction in (L.DIR_TOPDOWN, L.DIR_AUTO):
            dg.configure(launch=LAUNCHES[launch], direction=direction)
            for root in (0, 1, 599, 1199):
                _say(f"[gpu] deep caterpillar legs={legs} {launch} dir={direction} root={root}")
                st = _agrees(oracle, g, dg, root)
                if legs <= 14:
                    assert 1 < 4 * st["phases"] < st["levels"], st
                else:
                    assert st["phases"] >= st["levels"], st


@pytest.mark.parametrize("launch", list(LAUNCHES))
@pytest.mark.parametrize("branch,levels", [(3, 9), (7, 5), (15, 4)])
def test_deep_outgrown(oracle, branch, levels, launch):
    """A path into a tree, for each row form: the search is handed over on the
    path, outgrows a block's queue in the tree and starts again, the next ones
    stay in the ordinary form, also on another handle."""
    g = _padded(_path_then_tree(40, branch, levels))
    assert np.diff(g.beg_pos).max() == branch + 1
    with DeviceGraph(g) as dg, DeviceGraph(share=dg) as other:
        for h in (dg, other):
            h.configure(launch=LAUNCHES[launch], direction=L.DIR_TOPDOWN)
            for root in (0, 20, 0):
                _say(f"[gpu] deep outgrown branch={branch} {launch} root={root}")
                st = _agrees(oracle, g, h, root)
        assert st["phases"] >= st["levels"], st


def test_deep_directed_topdown_large(oracle):
    """Forced top-down on a directed ring with chords and vertices that have
    in-edges only, too many for one block."""
    n, ring = 17000, 600
    beg, adj = [0], []
    for v in range(n):
        row = sorted({(v + 1) % ring, ring + v * 20 % (n - ring)} | ({(v + 7) % ring} if v % 3 == 0 else set())) \
            if v < ring else []
        adj += row
        beg.append(len(adj))
    g = HostGraph.from_arrays(np.array(beg, np.int64), np.array(adj, np.int32))
    with DeviceGraph(g, keep_order=True) as dg:
        dg.configure(direction=L.DIR_TOPDOWN)
        for r in (0, 1, ring - 1):
            _say(f"[gpu] deep directed, large, root={r}")
            st = _agrees(oracle, g, dg, r)
            assert 1 < 2 * st["phases"] < st["levels"], st
