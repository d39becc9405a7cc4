"""GPU edge-list to CSR construction (include/ent_convert.h) against the
oracle: every flag combination bit for bit (offsets, adjacency, weights),
the raw R-MAT tuples against the host generator's CSR, the ent_convert CLI
against the reference converter's committed outputs, and BFS on a handle
built from tuples."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from enterprise_amd import DeviceGraph, EntError, HostGraph
from enterprise_amd import _lib as L
from enterprise_amd import convert

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
GOLD = os.path.join(HERE, "golden", "convert")
CLI = os.path.join(ROOT, "enterprise_amd", "bin", "ent_convert")


def _say(msg):
    print(msg, flush=True)


def _tuples(seed, n, ne):
    rng = np.random.default_rng(seed)
    src = rng.integers(0, n, ne).astype(np.int32)
    dst = rng.integers(0, n, ne).astype(np.int32)
    dup = rng.integers(0, max(ne, 1), ne // 6)
    if ne:
        src, dst = np.concatenate([src, src[dup]]), np.concatenate([dst, dst[dup]])
    return src, dst


@pytest.mark.parametrize("flags", list(range(16)))
@pytest.mark.parametrize("n,ne,seed", [(1, 0, 0), (1, 5, 1), (7, 30, 2), (300, 2000, 3), (5000, 40000, 4)])
def test_build_matches_oracle(oracle, flags, n, ne, seed):
    src, dst = _tuples(seed, n, ne)
    w = np.random.default_rng(seed + 99).integers(1, 64, src.size).astype(np.int32)
    _say(f"[gpu] csr_build n={n} ne={src.size} flags={flags}")
    g, wo, st = convert.csr_build(n, src, dst, flags, weight=w)
    b, a, ww = oracle.csr_build(n, src, dst, flags, weight=w)
    assert np.array_equal(g.beg_pos, b), (flags, n)
    assert np.array_equal(g.adj, a), (flags, n)
    assert np.array_equal(wo, ww), (flags, n)
    assert st["m"] == a.size and st["records"] == src.size * (2 if flags & L.CSR_REVERSE else 1)
    # Without weights the sorted forms sort keys alone: same CSR.
    g2, _, _ = convert.csr_build(n, src, dst, flags)
    assert np.array_equal(g2.beg_pos, b) and np.array_equal(g2.adj, a)


def test_build_large_ids_and_isolated_runs(oracle):
    """Ids at both ends of n = 2^30 + 12345 (runs of a billion empty rows,
    filled by the gap kernel) and a 62-bit sort key."""
    n = (1 << 30) + 12345
    rng = np.random.default_rng(8)
    src = (n - 1 - rng.integers(0, 1000, 3000)).astype(np.int32)
    dst = (n - 1 - rng.integers(0, 1000, 3000)).astype(np.int32)
    src[:10] = np.arange(10)
    dst[10:20] = np.arange(500, 510)
    _say("[gpu] csr_build n=2^30+12345")
    for flags in (L.CSR_SIMPLE, L.CSR_REVERSE):
        g, _, st = convert.csr_build(n, src, dst, flags)
        assert st["key_bits"] == (62 if flags & L.CSR_DEDUP else 31)
        # Against the oracle on relabelled ids (its offsets would need 8 GiB).
        ids = np.unique(np.concatenate([src, dst]))
        rs, rd = np.searchsorted(ids, src).astype(np.int32), np.searchsorted(ids, dst).astype(np.int32)
        wb, wa, _ = oracle.csr_build(ids.size, rs, rd, flags)
        b = g.beg_pos
        assert np.array_equal(b[ids], wb[:-1]) and b[-1] == wb[-1] == g.m
        assert np.array_equal(g.adj, ids[wa].astype(np.int32))
        # Offsets of the empty rows between the touched ones.
        assert np.array_equal(b[np.arange(0, n + 1, 1 << 20)], wb[np.searchsorted(ids, np.arange(0, n + 1, 1 << 20))])


def test_bad_tuples_rejected():
    with pytest.raises(EntError) as e:
        convert.csr_build(10, np.array([1, 10], np.int32), np.array([2, 3], np.int32), 0)
    assert e.value.code == L.ENT_EINVAL
    with pytest.raises(EntError) as e:
        convert.csr_build(10, np.array([1], np.int32), np.array([2], np.int32), 64)
    assert e.value.code == L.ENT_EINVAL


@pytest.mark.parametrize("scale", [16, 20])
def test_rmat_tuples_build_generator_graph(scale):
    """Size-independent property at scale 20: the device build of the raw
    tuples equals the host generator's CSR."""
    src, dst = convert.rmat_tuples(scale, 16, seed=scale)
    _say(f"[gpu] rmat tuples scale {scale}")
    g, _, st = convert.csr_build(1 << scale, src, dst, L.CSR_SIMPLE)
    h = HostGraph.rmat(scale, 16, seed=scale)
    assert np.array_equal(g.beg_pos, h.beg_pos) and np.array_equal(g.adj, h.adj)
    assert st["device_ms"] > 0


def test_build_device_arrays(oracle):
    """ent_csr_build_device on device-resident arrays."""
    src, dst = _tuples(12, 4000, 30000)
    h = HostGraph.rmat(8, 4, seed=1)
    with DeviceGraph(h) as dg:
        ne = src.size
        ps, pd = dg.device_alloc(4 * ne), dg.device_alloc(4 * ne)
        pb, pa = dg.device_alloc(8 * 4001), dg.device_alloc(4 * 2 * ne)
        try:
            import ctypes as C
            hip = C.CDLL("libamdhip64.so")
            hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
            assert hip.hipMemcpy(ps, src.ctypes.data, 4 * ne, 1) == 0
            assert hip.hipMemcpy(pd, dst.ctypes.data, 4 * ne, 1) == 0
            m, st = convert.csr_build_device(4000, ne, ps, pd, L.CSR_SIMPLE, pb, pa, 2 * ne)
            b = np.empty(4001, np.int64)
            a = np.empty(m, np.int32)
            assert hip.hipMemcpy(b.ctypes.data, pb, 8 * 4001, 2) == 0
            assert hip.hipMemcpy(a.ctypes.data, pa, 4 * m, 2) == 0
        finally:
            for p in (ps, pd, pb, pa):
                dg.device_free(p)
    wb, wa, _ = oracle.csr_build(4000, src, dst, L.CSR_SIMPLE)
    assert np.array_equal(b, wb) and np.array_equal(a, wa) and st["m"] == m


@pytest.mark.parametrize("reverse", [0, 1])
def test_cli_matches_reference_outputs(tmp_path, reverse):
    text = open(os.path.join(GOLD, "tuples.txt")).read()
    p = tmp_path / "t.txt"
    p.write_text(text)
    _say(f"[gpu] ent_convert reverse={reverse}")
    r = subprocess.run([CLI, str(p), str(reverse), "2"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    ref = np.load(os.path.join(GOLD, f"ref_rev{reverse}.npz"))
    got = {k: np.fromfile(f"{p}_{k}.bin", dtype=np.int64) for k in ("beg_pos", "csr", "deg", "head", "weight")}
    for k in ("beg_pos", "csr", "deg", "weight"):
        assert np.array_equal(got[k], ref[k]), k
    rows = np.repeat(np.arange(got["beg_pos"].size - 1), np.diff(got["beg_pos"]))
    assert np.array_equal(got["head"], rows)
    # The files load as a graph through the reference's binary format.
    g = HostGraph.read_bin(f"{p}_beg_pos.bin", f"{p}_csr.bin")
    assert g.m == ref["csr"].size


def test_cli_simple_graph_options(oracle, tmp_path):
    text = "1 2\n2 2\n2 3\n1 2\n3 1\n"
    p = tmp_path / "s.txt"
    p.write_text(text)
    r = subprocess.run([CLI, str(p), "1", "0", "--no-loops", "--dedup", "--out", str(tmp_path / "o")],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    g = HostGraph.read_bin(tmp_path / "o_beg_pos.bin", tmp_path / "o_csr.bin")
    b, a, _ = oracle.csr_build(3, [0, 1, 1, 0, 2], [1, 1, 2, 1, 0], L.CSR_SIMPLE)
    assert np.array_equal(g.beg_pos, b) and np.array_equal(g.adj, a)


def test_upload_edges_bfs(oracle):
    """A BFS handle built from tuples gives the oracle's depths on the host
    generator's graph."""
    src, dst = convert.rmat_tuples(14, 16, seed=14)
    h = HostGraph.rmat(14, 16, seed=14)
    with DeviceGraph.from_edges(1 << 14, src, dst) as dg:
        assert dg.m == h.m
        for r in h.pick_roots(4, 77):
            got, _ = dg.bfs(int(r))
            assert np.array_equal(got, oracle.bfs(h.beg_pos, h.adj, int(r))), r


def _one_row(n, ne, seed):
    """Every tuple in row 0 (one leaf holds them all), columns repeating."""
    rng = np.random.default_rng(seed)
    return np.zeros(ne, np.int32), rng.integers(0, n, ne).astype(np.int32)


PARTITION_CASES = {
    # Largest leaf of each sort kernel, one record less and more, and merged
    # leaves of 2, 3 and 7 chunks (odd and even numbers of merge passes).
    **{f"row0_{ne}": (lambda ne=ne: (1000, *_one_row(1000, ne, ne)))
       for ne in (1, 2, 63, 64, 65, 4095, 4096, 4097, 16383, 16384, 16385, 32769, 49153, 100001)},
    # A hub among ordinary rows, its columns spread over 2^20 ids.
    "hub": lambda: (1 << 20, *(np.concatenate(x) for x in zip(_one_row(1 << 20, 70000, 5), _tuples(6, 1 << 20, 50000)))),
    # Tile edges of the partition passes.
    **{f"tile_{ne}": (lambda ne=ne: (5000, *_tuples(ne, 5000, ne)))
       for ne in (3510, 3511, 4095, 4096, 4097, 8191, 8192, 8193)},
    # One pass and two, every vertex count around a power of two.
    **{f"n_{n}": (lambda n=n: (n, *_tuples(n, n, 20000)))
       for n in (1, 2, 255, 256, 257, 65535, 65536, 65537, (1 << 20) + 1, 1 << 22, (1 << 23) + 5, 1 << 24,
                 (1 << 24) + 1)},
    # Columns close together in an id range of 2^20: bins above their limit.
    **{f"crowded_{ne}": (lambda ne=ne: (1 << 20, *(np.concatenate(x) for x in zip(
        _one_row(512, ne, ne), _tuples(9, 1 << 20, 9000))))) for ne in (700, 9000, 16384, 40000)},
    "two_passes": lambda: (1 << 16, *_tuples(3, 1 << 16, 1200000)),
}


@pytest.mark.parametrize("case", list(PARTITION_CASES))
def test_sorted_rows_by_partition(oracle, case):
    """Sorted rows without weights at the edges of the partition build (leaf
    and tile sizes, passes, key widths; the largest n takes the radix sort):
    the oracle's CSR, bit for bit."""
    n, src, dst = PARTITION_CASES[case]()
    for flags in (L.CSR_SORT, L.CSR_SORT | L.CSR_REVERSE, L.CSR_DEDUP | L.CSR_NO_LOOPS, L.CSR_SIMPLE):
        _say(f"[gpu] csr_build {case} n={n} ne={src.size} flags={flags}")
        g, _, st = convert.csr_build(n, src, dst, flags)
        b, a, _ = oracle.csr_build(n, src, dst, flags)
        assert np.array_equal(g.beg_pos, b) and np.array_equal(g.adj, a), flags
        assert st["m"] == a.size


def test_partition_drops_every_record():
    """Loops alone, all dropped: an empty CSR."""
    ids = np.arange(3000, dtype=np.int32)
    g, _, st = convert.csr_build(3000, ids, ids, L.CSR_SIMPLE)
    assert g.m == 0 and st["m"] == 0 and not g.beg_pos.any()


def test_scratch_is_kept_and_given_back():
    """The scratch of a construction serves the next one, and goes back when
    the program asks for it and when a handle of the device is freed."""
    kept = L.lib().ent_internal_scratch_bytes
    kept.argtypes, kept.restype = [C.c_int32], C.c_int64
    src, dst = _tuples(17, 1 << 16, 200000)

    def build(tuples):
        g, _, _ = convert.csr_build(1 << 16, src[:tuples], dst[:tuples], convert.SIMPLE)
        return g.m

    convert.release_scratch()
    assert kept(0) == 0
    for give_back in (convert.release_scratch, lambda: DeviceGraph(HostGraph.rmat(8, 4, seed=1)).free()):
        _say("[gpu] construction scratch")
        m = build(src.size)
        size = kept(0)
        assert 8 * 2 * src.size < size < 1 << 30  # more than the records' keys
        assert build(src.size) == m and kept(0) == size
        build(1000)  # a smaller one runs in the same block
        assert kept(0) == size
        give_back()
        assert kept(0) == 0
    convert.release_scratch()  # nothing left: no error
    for device in (-1, 1 << 20):
        with pytest.raises(EntError):
            convert.release_scratch(device)


def test_builds_of_different_sizes_at_once(oracle):
    """Four threads whose histograms take 4 bytes to 128 KiB of LDS: what one
    asks of the runtime for its launch is no limit for another's."""
    import threading
    wrong = []

    def work(n, ne, seed):
        try:
            for i in range(10):
                src, dst = _tuples(1000 * seed + i, n, ne)
                g, _, _ = convert.csr_build(n, src, dst, L.CSR_SORT)
                b, a, _ = oracle.csr_build(n, src, dst, L.CSR_SORT)
                if not (np.array_equal(g.beg_pos, b) and np.array_equal(g.adj, a)):
                    wrong.append((n, i))
        except Exception as e:  # an error in a thread fails the test
            wrong.append((n, e))

    threads = [threading.Thread(target=work, args=x)
               for x in ((1 << 24, 3000, 1), (1, 10, 2), (10, 100, 3), (1 << 22, 20000, 4))]
    _say("[gpu] csr_build in four threads")
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:3]


def _sorted_csr(n, src, dst, reverse, dedup):
    """The CSR by one sort of 64-bit keys on the device, torch's."""
    import torch
    u, v = src.long(), dst.long()
    key = u * n + v
    if reverse:
        key = torch.cat([key, v * n + u])
    key = torch.unique(key) if dedup else torch.sort(key).values
    beg = torch.searchsorted(torch.div(key, n, rounding_mode="floor"), torch.arange(n + 1, device="cuda"))
    return beg, (key % n).int()


@pytest.mark.parametrize("share", [0.0, 0.2, 0.35, 1.0])
@pytest.mark.parametrize("rows", [3000, 1 << 18])
def test_long_row_turns_to_radix(rows, share):
    """2^24 records and one row with a share of the tuples: on both sides of
    the share at which a large build leaves the partition for the radix sort
    (3 of 9 merge passes at 2^23 records, a third of the forward half). A
    second build in the same scratch follows each."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(rows + int(100 * share))
    ne = 1 << 24
    src, dst = (torch.randint(0, rows, (ne,), generator=gen, device="cuda", dtype=torch.int32) for _ in range(2))
    src[torch.rand(ne, generator=gen, device="cuda") < share] = 7
    for flags, tuples in ((L.CSR_SORT, ne), (L.CSR_SORT | L.CSR_REVERSE, ne // 2), (L.CSR_DEDUP | L.CSR_REVERSE, ne // 2),
                          (L.CSR_SORT, 5000)):
        s, d = src[:tuples].contiguous(), dst[:tuples].contiguous()
        rev = bool(flags & L.CSR_REVERSE)
        beg = torch.empty(rows + 1, dtype=torch.int64, device="cuda")
        adj = torch.empty(tuples * (2 if rev else 1), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        _say(f"[gpu] csr_build, one row with {share} of {tuples} tuples, {rows} rows, flags={flags}")
        m, _ = convert.csr_build_device(rows, tuples, s.data_ptr(), d.data_ptr(), flags, beg.data_ptr(), adj.data_ptr(),
                                        adj.numel())
        want_beg, want_adj = _sorted_csr(rows, s, d, rev, bool(flags & L.CSR_DEDUP))
        assert m == want_adj.numel()
        assert torch.equal(beg, want_beg) and torch.equal(adj[:m], want_adj), flags


@pytest.mark.parametrize("rows,ne", [(1, 131071), (1, 131072), (2, 262143), (2, 262144), (64, 8 << 20), (64, (8 << 20) - 1)])
def test_few_rows(rows, ne):
    """Both sides of eight chunks a row, from where the radix sort is taken."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(ne)
    src, dst = (torch.randint(0, rows, (ne,), generator=gen, device="cuda", dtype=torch.int32) for _ in range(2))
    beg = torch.empty(rows + 1, dtype=torch.int64, device="cuda")
    adj = torch.empty(ne, dtype=torch.int32, device="cuda")
    for flags in (L.CSR_SORT, L.CSR_DEDUP):
        torch.cuda.synchronize()
        _say(f"[gpu] csr_build, {rows} rows, {ne} tuples, flags={flags}")
        m, _ = convert.csr_build_device(rows, ne, src.data_ptr(), dst.data_ptr(), flags, beg.data_ptr(), adj.data_ptr(), ne)
        want_beg, want_adj = _sorted_csr(rows, src, dst, False, bool(flags & L.CSR_DEDUP))
        assert m == want_adj.numel()
        assert torch.equal(beg, want_beg) and torch.equal(adj[:m], want_adj), flags
