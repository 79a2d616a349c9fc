"""Row splits and component folds at the sizes where they change: rows at and
around the lane / 16-lane / chunk limits in the 64-source pull, and component
minima over a giant component, pairs and isolated vertices."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
G = pytest.importorskip("graptor_amd")


@pytest.fixture(scope="module", autouse=True)
def device():
    G.lib()
    yield


# rows at the limits of the lane (32), 16-lane (2048) and chunk (8192) splits
HUBS = (1, 31, 32, 33, 64, 65, 2047, 2048, 2049, 8191, 8192, 8193, 16400)


def hub_graph(n):
    """Vertex i < len(HUBS) has edges to HUBS[i] later vertices; the others hang off them."""
    src, dst = [], []
    for i, d in enumerate(HUBS):
        src.append(np.full(d, i, np.uint32))
        dst.append((len(HUBS) + (np.arange(d) * 7 + i) % (n - len(HUBS))).astype(np.uint32))
    return O.build_csr(n, np.concatenate(src), np.concatenate(dst))


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("k", [1, 15, 16, 17, 63, 64])
def test_msbfs_pull_row_lengths(k, reorder):
    n = 25013
    index, nbrs = hub_graph(n)
    src = (np.arange(k, dtype=np.uint32) * 389) % n
    with G.Graph.from_csr(index, nbrs) as g:
        if reorder:
            g.reorder()
        ref = O.msbfs_levels(index, nbrs, src)
        for d in (G.DIR_PULL, G.DIR_AUTO):
            lv, _ = g.msbfs(src, direction=d)
            assert np.array_equal(lv, ref), d


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("n", [1, 2, 63, 257, 2049, 70001])
def test_component_minima(n, reorder):
    # a chain over the odd vertices (one giant component that starts at 1),
    # pairs among the multiples of 8, the other even vertices alone
    v = np.arange(n, dtype=np.uint32)
    odd = v[v % 2 == 1]
    pair = v[(v % 16 == 0) & (v + 8 < n)]
    src = np.concatenate((odd[:-1], pair)) if len(odd) else pair
    dst = np.concatenate((odd[1:], pair + 8)) if len(odd) else pair + 8
    index, nbrs = O.build_csr(n, src.astype(np.uint32), dst.astype(np.uint32))
    with G.Graph.from_csr(index, nbrs) as g:
        if reorder:
            g.reorder()
        lab, _ = g.ccv()
    assert np.array_equal(lab, O.cc_labels(index, nbrs))


def test_component_minima_two_giants():
    # two interleaved giants: every wave meets both labels
    n = 300007
    v = np.arange(n - 2, dtype=np.uint32)
    index, nbrs = O.build_csr(n, v, v + 2)
    with G.Graph.from_csr(index, nbrs) as g:
        p = g.prop()
        p.upload((np.arange(n) % 2).astype(np.uint32))
        out = np.empty(n, np.uint32)
        G._check(G.lib().gpr_cc_recode(p.h, out.ctypes.data))
        p.destroy()
    assert np.array_equal(out, (np.arange(n) % 2).astype(np.uint32))


@pytest.mark.parametrize("n", [700, 5003, 60013])
@pytest.mark.parametrize("d", [2, 8, 30, 32, 34, 256, 258])
def test_kcore_regular_rows(n, d):
    """A ring where every vertex has d neighbours, and a pendant path: rows at
    the lane and slice limits in rounds of few and of many vertices (one round
    peels the whole ring)."""
    v = np.arange(n, dtype=np.uint32)
    src = [np.repeat(v, d // 2)]
    dst = [((src[0] + np.tile(np.arange(1, d // 2 + 1), n)) % n).astype(np.uint32)]
    tail = np.arange(n, n + 40, dtype=np.uint32)
    src.append(np.concatenate((np.zeros(1, np.uint32), tail[:-1])))
    dst.append(tail)
    index, nbrs = O.build_csr(n + 40, np.concatenate(src), np.concatenate(dst))
    for reorder in (False, True):
        with G.Graph.from_csr(index, nbrs) as g:
            if reorder:
                g.reorder()
            core, kmax, info = g.kcore()
        assert kmax == d and (core[:n] == d).all() and (core[n:] == 1).all()
        assert info.edges == len(nbrs)


def ring(n, reach, gap=0):
    """Vertex i joined to the next `reach` ones around a ring; 0 is a cut-off vertex if gap."""
    i = np.repeat(np.arange(gap, n), reach)
    j = gap + (i - gap + np.tile(np.arange(1, reach + 1), n - gap)) % (n - gap)
    return i.astype(np.uint32), j.astype(np.uint32)


def test_batch_cc_row_runs():
    """Graphs around the 64-vertex runs, the runs left to all waves (more of
    them than are kept, and single rows of a whole run's edges) and the size
    whose parents fit on chip."""
    parts = [(n, ring(n, 1, 1)) for n in (3, 63, 64, 65, 127, 128, 129)]
    for n in (64, 4096, 4097, 4098, 65536, 65537):   # stars: rows of 63 .. 65536 edges
        hub = n - 1 if n % 2 else 0
        leaf = np.delete(np.arange(n, dtype=np.uint32), hub)
        parts.append((n, (np.full(n - 1, hub, np.uint32), leaf)))
    parts.append((5000, ring(5000, 40, 1)))          # 79 runs of 5120 edges
    parts.append((2, (np.zeros(0, np.uint32), np.zeros(0, np.uint32))))
    voff, src, dst, n = [0], [], [], 0
    for k, (a, b) in parts:
        src.append(n + a)
        dst.append(n + b)
        n += k
        voff.append(n)
    index, nbrs = O.build_csr(n, np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32))
    with G.Batch.from_csr(index, nbrs, np.array(voff, np.uint32)) as b:
        lab, _ = b.cc()
    assert np.array_equal(lab, O.cc_labels(index, nbrs))


@pytest.mark.parametrize("n", [1, 64, 1024, 1025, 16385, 655361, 2 * 1048576 + 1026])
def test_bitmap_to_list_and_degree_prefix(n):
    """Per-workgroup counts scanned by the last workgroup: one, several, a thread's share (8) of each thread and
    more (1024 list entries and 16384 bits a workgroup)."""
    leaf = np.arange(1, n, dtype=np.uint32)
    index, nbrs = O.build_csr(n, np.zeros(n - 1, np.uint32), leaf) if n > 1 else (
        np.zeros(2, np.uint64), np.zeros(0, np.uint32))
    with G.Graph.from_csr(index, nbrs) as g:
        for every in (1, 3, 1000):
            want = np.arange(0, n, every, dtype=np.uint32)
            f = G.Frontier(g)
            f.set_list(want)
            f.convert(G.FRONTIER_BITMAP)
            f.convert(G.FRONTIER_LIST)
            assert f.stats()[:2] == (len(want), int(np.diff(index)[want].sum()))
            assert np.array_equal(f.download(), want)
            f.destroy()
        # from a leaf: the hub, then a list of all other leaves
        lv, _ = g.bfslvl(n - 1, direction=G.DIR_PUSH)
        assert np.array_equal(lv, O.bfs_levels(index, nbrs, n - 1))
