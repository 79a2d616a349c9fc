"""Results into every kind of buffer that the runtime's copies take: pageable
memory, pinned memory, a part of a pinned block that is too small for them, and
device memory; small graphs and large, more than once a handle."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
G = pytest.importorskip("graptor_amd")
torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True)
def device():
    G.lib()


@pytest.mark.parametrize("where", ["pageable", "pinned", "device"])
@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("n", [70, 4099, 300007])
def test_results_reach_the_buffer(n, reorder, where):
    k = np.arange(3 * n, dtype=np.uint64)
    index, nbrs = O.build_csr(n, (k * 7919 % n).astype(np.uint32), (k * k * 31 % n).astype(np.uint32))
    levels, labels = O.bfs_levels(index, nbrs, 1), O.cc_labels(index, nbrs)
    t = torch.zeros(n, dtype=torch.int32, device="cuda" if where == "device" else "cpu", pin_memory=where == "pinned")
    torch.cuda.synchronize()
    dst, info = C.c_void_p(t.data_ptr()), G.RunInfo()

    def got():
        v = t.cpu().numpy().view(np.uint32).copy()
        t.zero_()
        torch.cuda.synchronize()
        return v

    with G.Graph.from_csr(index, nbrs) as g:
        if reorder:
            g.reorder()
        for o in (None, None, None, G.opts(direction=G.DIR_PUSH)):    # whole runs, then a driven one
            G._check(G.lib().gpr_bfslvl(g.h, 1, o and C.byref(o), dst, C.byref(info)))
            assert np.array_equal(got(), levels)
            G._check(G.lib().gpr_ccv(g.h, o and C.byref(o), dst, C.byref(info)))
            assert np.array_equal(got(), labels)
