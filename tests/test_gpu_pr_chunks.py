"""PageRank's binned edgemap where its tiles and chunks change with the graph:
sizes around one bin (16384), one tile (1024), bins in one chunk, in up to a
group of 16 and in several groups, directed and relabelled graphs; and where
the rule for small graphs (pr_pull_edges) pulls instead.

Bars as in test_gpu_pr_split: relative L1 against FP64 of 1e-6 for FP32 (each
rank is rounded to 24 bits a few times an iteration, and errors contract by
the damping) and 1e-3 for 16-bit contributions on power-law graphs; repeated
runs are bit-identical.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
G = pytest.importorskip("graptor_amd")


@pytest.fixture(scope="module", autouse=True)
def device():
    G.lib()
    old = G.tune_get("pr_pull_edges")
    yield
    G.tune_set("pr_pull_edges", old)


def rel_l1(a, b):
    return float(np.abs(a.astype(np.float64) - b).sum() / np.abs(b).sum())


def skewed(n, m, seed):
    """m directed edges whose ends follow a power law over n vertices."""
    rng = np.random.default_rng(seed)
    return tuple((n * rng.random(m) ** 3).astype(np.uint32) for _ in range(2))


# vertices, edges drawn: one bin or tile more or less, few and many chunks
SIZES = [(1023, 4000), (1025, 60000), (16383, 40000), (16385, 300000), (40001, 1500000), (70003, 6000000),
         (600011, 3000000)]


@pytest.mark.parametrize("n,m", SIZES)
@pytest.mark.parametrize("directed", [False, True])
@pytest.mark.parametrize("pull", [0, 1 << 23])
def test_ranks_across_layout_sizes(n, m, directed, pull):
    G.tune_set("pr_pull_edges", pull)   # 0: every edge binned
    src, dst = skewed(n, m, n)
    index, nbrs = O.build_csr(n, src, dst, symmetrize=not directed)
    if directed:
        ci, cn = O.build_csr(n, dst, src, symmetrize=False)
        x64, _, _ = O.pr_fp64(ci, cn, 12, 0.0, outdeg=np.diff(index).astype(np.uint32))
    else:
        x64, _, _ = O.pr_fp64(index, nbrs, 12, 0.0)
    with G.Graph.from_csr(index, nbrs, symmetric=not directed) as g:
        if not directed:
            g.reorder()
        for fmt, bar in (("fp32", 1e-6), ("fp16", 1e-3)):
            x, _ = g.pr_vary([(fmt, 0.0)], max_iter=12)
            assert rel_l1(x, x64) <= bar, (fmt, rel_l1(x, x64))
            x2, _ = g.pr_vary([(fmt, 0.0)], max_iter=12)
            assert np.array_equal(x, x2), fmt


@pytest.mark.parametrize("fmt", ["fp32", "bf16", "fp16", "cfp16", "scfp16"])
@pytest.mark.parametrize("pull", [0, 1 << 23])
def test_fused_iterations_equal_unfused(fmt, pull):
    """A fixed iteration count (tails fused into the next iteration) and a
    convergence test that never stops the run give the same ranks."""
    G.tune_set("pr_pull_edges", pull)
    n = 30011
    src, dst = skewed(n, 400000, 3)
    index, nbrs = O.build_csr(n, src, dst)
    with G.Graph.from_csr(index, nbrs).reorder() as g:
        xf, _ = g.pr_vary([(fmt, 0.0)], max_iter=9)
        xu, _ = g.pr_vary([(fmt, 1e-300)], max_iter=9)
    assert np.array_equal(xf.view(np.uint32), xu.view(np.uint32))


@pytest.mark.parametrize("hubs,degree", [(1, 2049), (255, 2100), (256, 2100), (257, 2100), (1, 256 * 8192), (1, 257 * 8192)])
def test_long_rows_folded_in_the_pull(hubs, degree):
    """Rows in as many chunks (8192 edges) as the pull's last workgroup folds, and in more."""
    n = max(4001, degree + hubs)
    dst = np.repeat(np.arange(hubs, dtype=np.uint32), degree)
    src = (hubs + (np.arange(hubs * degree, dtype=np.uint64) * 7 + dst) % (n - hubs)).astype(np.uint32)
    back = np.arange(n, dtype=np.uint32)     # every vertex has a way on
    src, dst = np.concatenate([src, back]), np.concatenate([dst, (back * 31 + 7) % n])
    index, nbrs = O.build_csr(n, src, dst.astype(np.uint32), symmetrize=False)
    ci, cn = O.build_csr(n, dst.astype(np.uint32), src, symmetrize=False)
    x64, _, _ = O.pr_fp64(ci, cn, 8, 0.0, outdeg=np.diff(index).astype(np.uint32))
    with G.Graph.from_csr(index, nbrs, symmetric=False) as g:
        for fmt, bar in (("fp32", 1e-6), ("fp16", 1e-3)):
            x, _ = g.pr_vary([(fmt, 0.0)], max_iter=8)
            assert rel_l1(x, x64) <= bar, (fmt, rel_l1(x, x64))
            x2, _ = g.pr_vary([(fmt, 0.0)], max_iter=8)
            assert np.array_equal(x, x2), fmt
