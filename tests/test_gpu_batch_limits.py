"""gpr_batch_cc_noalloc on batches that its host side cannot check: vertex
ranges that overlap.  The labels of such a batch are not defined; the call
returns, writes labels that are vertices of the batch, and leaves the next
batch's labels right."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
G = pytest.importorskip("graptor_amd")
torch = pytest.importorskip("torch")


def noalloc(index, nbrs, voff):
    n = len(index) - 1
    ix, nb, vo = (torch.from_numpy(np.ascontiguousarray(a).view(t)).cuda()
                  for a, t in ((index, np.int64), (nbrs, np.int32), (voff, np.int32)))
    lab = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    G._check(G.lib().gpr_batch_cc_noalloc(ix.data_ptr(), nb.data_ptr(), vo.data_ptr(), len(voff) - 1, n,
                                          lab.data_ptr(), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    return lab.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("voff", [
    [0, 150000, 70000, 300000, 100000, 400000],             # three graphs that share ranges
    [100000, 300000, 0, 200000, 50000, 250000, 130000, 400000],
    [0, 400000, 0, 400000, 0, 400000, 0, 400000],           # the same one four times
])
def test_overlapping_large_graphs(voff):
    G.lib()
    n = 400000
    rng = np.random.default_rng(5)
    index, nbrs = O.build_csr(n, rng.integers(0, n, 900000).astype(np.uint32), rng.integers(0, n, 900000).astype(np.uint32))
    voff = np.array(voff, np.uint32)
    lab = noalloc(index, nbrs, voff)
    covered = np.zeros(n, bool)
    for a, b in zip(voff[:-1], voff[1:]):
        covered[a:max(a, b)] = True
    assert (lab[covered] < n).all() and (lab[~covered] == 0xFFFFFFFF).all()
    assert (lab[covered] <= np.arange(n)[covered]).all()
    two = np.array([0, 180000, n], np.uint32)
    cut = np.repeat(np.arange(n), np.diff(index).astype(np.int64)) < 180000
    same = cut == (nbrs < 180000)
    src = np.repeat(np.arange(n, dtype=np.uint32), np.diff(index).astype(np.int64))[same]
    ix, nb = O.build_csr(n, src, nbrs[same], symmetrize=False)
    assert np.array_equal(noalloc(ix, nb, two), O.cc_labels(ix, nb))
