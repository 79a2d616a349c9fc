"""PageRank's binned edgemap on graphs that the default rule (pr_pull_edges)
pulls: the split tests and delta PageRank's, with every edge that they bin
really binned; and tiles that their edge count closes, under tiles as wide as
the graph's size makes them."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
G = pytest.importorskip("graptor_amd")

import test_gpu_apr as apr                                                            # noqa: E402
from test_gpu_pr_split import (rel_l1, restore_split, split_at,                       # noqa: E402,F401
                               test_fused_tail_iteration_bit_identical, test_prv_fused_tail_equals_unfused,
                               test_split_converged_stages, test_split_directed_graph, test_split_formats_vs_fp64,
                               test_split_fp32_vs_fp64_and_unsplit, test_split_point_changes_and_graph_reuse,
                               test_split_rmat20_chunked_hub_bins, test_write_run_offsets_from_hbm)


@pytest.fixture(autouse=True)
def binned(monkeypatch):
    """pr_pull_edges 0; after the test, that its handles ran the binned kernels."""
    G.lib()
    old = G.tune_get("pr_pull_edges")
    G.tune_set("pr_pull_edges", 0)
    ran = []
    create, destroy = G.Graph.__init__, G.Graph.destroy

    def profiled(self, *a):
        create(self, *a)
        self.profile()

    def counted(self):
        if self.h:
            ran.append(self.profile_get("pr_cold_write")[1])
        destroy(self)

    monkeypatch.setattr(G.Graph, "__init__", profiled)
    monkeypatch.setattr(G.Graph, "destroy", counted)
    yield
    G.tune_set("pr_pull_edges", old)
    assert sum(ran) > 0, "no binned kernel ran"


@pytest.mark.parametrize("name", sorted(apr.GRAPHS))
@pytest.mark.parametrize("variant", sorted(apr.STAGES))
def test_apr_matches_oracle(name, variant):
    (index, nbrs), sym = apr.GRAPHS[name]
    with G.Graph.from_csr(index, nbrs, symmetric=sym) as g:
        for d in (G.DIR_AUTO, G.DIR_PULL):
            apr.test_apr_matches_oracle((name, index, nbrs, sym, g), variant, d)


def ranks(g, split, iters):
    G.tune_set("pr_split_bytes", split)
    return g.prv(max_iter=iters)[0]


def check_against_pull(index, nbrs, x64, symmetric, iters):
    with G.Graph.from_csr(index, nbrs, symmetric=symmetric) as g:
        x0 = ranks(g, 1e12, iters)
        x1, x2 = ranks(g, 0.0, iters), ranks(g, 0.0, iters)
    assert np.array_equal(x1, x2)
    assert rel_l1(x1, x0) <= 5e-8, rel_l1(x1, x0)
    assert rel_l1(x1, x64) <= 1e-6, rel_l1(x1, x64)


def test_tile_closed_by_edge_count():
    """1024 consecutive sources, as wide as a small graph's tile, with 18.4M edges: the tile closes before its last
    source."""
    hubs, per, leaves = 1024, 18000, 40000
    h = np.arange(hubs, dtype=np.int64)
    src = np.concatenate((np.repeat(h, per), hubs + np.arange(leaves))).astype(np.uint32)
    dst = np.concatenate((hubs + (np.repeat(h * 37, per) + np.tile(np.arange(per), hubs)) % leaves,
                          np.arange(leaves) % hubs)).astype(np.uint32)
    index, nbrs = O.build_csr(hubs + leaves, src, dst, symmetrize=False)
    assert index[hubs] > 1 << 24 and index[hubs] == hubs * per
    ci, cn = O.build_csr(hubs + leaves, dst, src, symmetrize=False)
    x64, _, _ = O.pr_fp64(ci, cn, 8, 0.0, outdeg=np.diff(index).astype(np.uint32))
    check_against_pull(index, nbrs, x64, False, 8)


def test_one_source_above_the_edge_count():
    """A source with more edges than a tile takes has a tile of its own."""
    d = (1 << 24) + 100
    n = d + 3
    index = np.concatenate(([0], d + np.arange(d + 1), [2 * d, 2 * d])).astype(np.uint64)   # a star, two alone
    nbrs = np.concatenate((np.arange(1, d + 1), np.zeros(d))).astype(np.uint32)
    assert len(index) == n + 1 and index[-1] == len(nbrs)
    x64, _, _ = O.pr_fp64(index, nbrs, 4, 0.0)
    check_against_pull(index, nbrs, x64, True, 4)
