"""A graph's run buffers go from one run to the next: a new property is zero
whatever held its memory before, runs that alternate give what single runs
give, and a property may outlive its graph."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
G = pytest.importorskip("graptor_amd")


@pytest.fixture(scope="module", autouse=True)
def device():
    G.lib()
    yield


@pytest.mark.parametrize("dtype,np_dtype", [(G.U16, np.uint16), (G.U32, np.uint32), (G.F64, np.float64),
                                            (G.U64, np.uint64)])
@pytest.mark.parametrize("n", [1, 63, 5003])
def test_new_property_is_zero(n, dtype, np_dtype):
    index, nbrs = O.build_csr(n, np.arange(n - 1, dtype=np.uint32), np.arange(1, n, dtype=np.uint32))
    with G.Graph.from_csr(index, nbrs) as g:
        for _ in range(40):      # more than the blocks that are kept
            p = [G.Prop(g, dtype) for _ in range(3)]
            for q in p:
                assert not q.download().any()
                q.upload(np.full(n, 7, np_dtype))
            for q in p:
                q.destroy()


def test_alternating_runs_and_late_destroy():
    index, nbrs = O.rmat_graph(12, 8)
    n = len(index) - 1
    g = G.Graph.from_csr(index, nbrs)
    src = (np.arange(64, dtype=np.uint32) * 37) % n
    want_ms, want_cc = O.msbfs_levels(index, nbrs, src), O.cc_labels(index, nbrs)
    first = None
    for _ in range(3):
        assert np.array_equal(g.msbfs(src)[0], want_ms)
        assert np.array_equal(g.ccv()[0], want_cc)
        pr = g.prv(max_iter=10)[0]
        first = pr if first is None else first
        assert np.array_equal(pr, first)      # integer accumulation: the same bits
    late = G.Prop(g, G.U32)
    g.destroy()
    late.destroy()
