"""The PageRank edgemap's sums of 16-bit contributions keep what FP32 would
lose: rows of one 1 and many 2^-25, whose exact sums FP32 can hold, pulled and
binned, over every split of a row (a lane's, a wave's, chunks)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
G = pytest.importorskip("graptor_amd")

# codes of 1 and of 2^-25
CODES = {"bf16": (0x3F80, 0x3300), "bf16t": (0x3F80, 0x3300), "cfp16": (0xFC00, 0x9800), "scfp16": (0x7E00, 0x4C00)}
DEGREES = [1, 2, 33, 64, 65, 200, 2048, 2049, 8192, 8193, 30001]


@pytest.fixture(autouse=True)
def restore():
    G.lib()
    old = {k: G.tune_get(k) for k in ("pr_pull_edges", "pr_split_bytes")}
    yield
    for k, v in old.items():
        G.tune_set(k, v)


@pytest.mark.parametrize("pull,split", [(1 << 23, 0.0), (0, 0.0), (0, 1e12), (0, 4096.0)],
                         ids=["small_pulled", "binned", "pulled", "split"])
@pytest.mark.parametrize("fmt", sorted(CODES))
def test_rows_keep_small_terms(fmt, pull, split):
    G.tune_set("pr_pull_edges", pull)
    G.tune_set("pr_split_bytes", split)
    k = max(DEGREES)
    n = k + len(DEGREES)
    # source s (< k) points to the rows of more than s in-edges
    outdeg = np.array([sum(d > s for d in DEGREES) for s in range(k)] + [0] * len(DEGREES), np.uint64)
    index = np.concatenate(([0], np.cumsum(outdeg))).astype(np.uint64)
    nbrs = np.concatenate([[k + i for i, d in enumerate(DEGREES) if d > s] for s in range(k)]).astype(np.uint32)
    one, tiny = CODES[fmt]
    codes = np.full(n, tiny, np.uint16)
    codes[0] = one
    want = np.zeros(n, np.float32)
    want[k:] = [np.float32(1.0 + (d - 1) * 2.0 ** -25) for d in DEGREES]
    with G.Graph.from_csr(index, nbrs, symmetric=False) as g:
        y, c = g.prop(G.F32), g.prop(G.U16)
        c.upload(codes)
        g.edgemap(G.RELAX_PR_SUM, y, contrib=c, contrib_fmt=G.CONTRIB_NAMES[fmt], damping=0.85)
        assert np.array_equal(y.download(), want)
        y.destroy()
        c.destroy()
