"""BFS and CC runs that stay on the device from start to end (whole_edges),
against the oracle and, step counts included, against the host-driven loop:
rows at the lane and slice limits, hubs of many slices, isolated and
single vertices, directed graphs, long paths, results above and below the
pinned staging size."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
G = pytest.importorskip("graptor_amd")


@pytest.fixture(scope="module", autouse=True)
def device():
    G.lib()
    yield


@pytest.fixture(autouse=True)
def restore_tunables():
    old = {k: G.tune_get(k) for k in ("whole_edges",)}
    yield
    for k, v in old.items():
        G.tune_set(k, v)


def star(d, n):
    """Vertex 0 next to 1..d, a path behind them, the rest alone."""
    src = np.concatenate((np.zeros(d, np.uint32), np.arange(1, d, dtype=np.uint32)))
    dst = np.concatenate((np.arange(1, d + 1, dtype=np.uint32), np.arange(2, d + 1, dtype=np.uint32)))
    return O.build_csr(n, src, dst)


def graphs():
    out = {"one": O.build_csr(1, np.zeros(0, np.uint32), np.zeros(0, np.uint32)),
           "alone": O.build_csr(70, np.zeros(0, np.uint32), np.zeros(0, np.uint32)),
           "path": O.build_csr(3001, np.arange(3000, dtype=np.uint32), np.arange(1, 3001, dtype=np.uint32)),
           "grid_long": O.grid_graph(251, 187, 0.01, seed=5),
           "er_sparse": O.er_graph(50021, 2, seed=7),
           "er": O.er_graph(30011, 6, seed=8),
           "rmat12": O.rmat_graph(12),
           "rmat16": O.rmat_graph(16),
           "er_unstaged": O.er_graph(300007, 5, seed=9)}
    for d in (31, 32, 33, 255, 256, 257, 2048, 2049, 40000):
        out["star%d" % d] = star(d, d + 5)
    return out


GRAPHS = graphs()


def host_driven(f):
    G.tune_set("whole_edges", 0)
    try:
        return f()
    finally:
        G.tune_set("whole_edges", 1 << 24)


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_whole_bfs(name, reorder):
    index, nbrs = GRAPHS[name]
    n = len(index) - 1
    with G.Graph.from_csr(index, nbrs) as g:
        if reorder:
            g.reorder()
        for s in sorted({0, n // 2, n - 1, O.highest_degree_vertex(index)}):
            lv, info = g.bfslvl(s)
            assert np.array_equal(lv, O.bfs_levels(index, nbrs, s)), s
            want, winfo = host_driven(lambda: g.bfslvl(s))
            assert np.array_equal(lv, want)
            assert (info.iters, info.push_iters, info.edges) == (winfo.iters, winfo.push_iters, winfo.edges), s
            none, again = g.bfslvl(s, download=False)
            assert none is None and again.edges == info.edges


@pytest.mark.parametrize("pct", [1.0, 5.0, 40.0])
def test_whole_bfs_threshold(pct):
    index, nbrs = GRAPHS["rmat16"]
    with G.Graph.from_csr(index, nbrs) as g:
        _, a = g.bfslvl(5, threshold_pct=pct)
        _, b = host_driven(lambda: g.bfslvl(5, threshold_pct=pct))
    assert (a.iters, a.push_iters, a.edges) == (b.iters, b.push_iters, b.edges)


def test_whole_bfs_directed():
    rng = np.random.default_rng(4)
    n = 20011
    src = rng.integers(0, n, 90000).astype(np.uint32)
    dst = (n * rng.random(90000) ** 2).astype(np.uint32)
    index, nbrs = O.build_csr(n, src, dst, symmetrize=False)
    with G.Graph.from_csr(index, nbrs, symmetric=False) as g:
        for s in (0, 17, int(src[5])):
            lv, info = g.bfslvl(s)
            assert np.array_equal(lv, O.bfs_levels(index, nbrs, s))
            _, b = host_driven(lambda: g.bfslvl(s))
            assert (info.iters, info.push_iters, info.edges) == (b.iters, b.push_iters, b.edges)


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_whole_cc(name, reorder):
    index, nbrs = GRAPHS[name]
    with G.Graph.from_csr(index, nbrs) as g:
        if reorder:
            g.reorder()
        for _ in range(2):
            lab, info = g.ccv()
            assert np.array_equal(lab, O.cc_labels(index, nbrs))
            assert info.edges == len(nbrs)
        none, _ = g.ccv(download=False)
        assert none is None


@pytest.mark.parametrize("n", [30011, 300007])
def test_whole_cc_long_paths_relabelled(n):
    """Long paths into deep trees: late path-halving stores leave parents that are not yet roots."""
    k = np.arange(3 * n, dtype=np.uint64)
    index, nbrs = O.build_csr(n, (k * 7919 % n).astype(np.uint32), (k * k * 31 % n).astype(np.uint32))
    want = O.cc_labels(index, nbrs)
    with G.Graph.from_csr(index, nbrs) as g:
        g.reorder()
        for _ in range(10):
            assert np.array_equal(g.ccv()[0], want)


@pytest.mark.parametrize("reach", [1, 2, 3, 4, 8, 9, 15, 16, 17])
@pytest.mark.parametrize("n", [70, 4099, 33000])
def test_whole_bfs_lanes_per_row(n, reach):
    """Rows of 2 to 34 edges, in levels that leave lanes for 1 to 8 a row: a ring with a hub's worth of short cuts
    from the start."""
    i = np.repeat(np.arange(n), reach)
    j = (i + np.tile(np.arange(1, reach + 1), n)) % n
    cut = np.arange(1, n, max(1, n // 3000))
    index, nbrs = O.build_csr(n, np.concatenate([i, 0 * cut]).astype(np.uint32), np.concatenate([j, cut]).astype(np.uint32))
    with G.Graph.from_csr(index, nbrs) as g:
        for s in (0, n // 2):
            lv, info = g.bfslvl(s)
            assert np.array_equal(lv, O.bfs_levels(index, nbrs, s))
            _, b = host_driven(lambda: g.bfslvl(s))
            assert (info.iters, info.push_iters, info.edges) == (b.iters, b.push_iters, b.edges)
