"""gpr_batch_cc_noalloc at its limits.  Batches that its host side cannot
check, with vertex ranges that overlap: the labels are not defined; the call
returns, writes labels that are vertices of the batch, and leaves the next
batch's labels right.  And 64 vertices with more edges than 32 bits count."""
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


def test_rows_of_more_than_32_bits_of_edges():
    """All but a few of vertex 0's edges lead to vertex 1; the others lie where positions in 32 bits would end and
    behind."""
    G.lib()
    n, m = 100, (1 << 32) + 1000
    if torch.cuda.mem_get_info()[0] < 5 * m:
        pytest.skip("needs 20 GB of device memory")
    nb = torch.ones(m, dtype=torch.int32, device="cuda")
    for k, at in enumerate((0xFFF00000 - 1, 0xFFF00000, 0xFFF00000 + 5, (1 << 32) - 1, 1 << 32, m - 1)):
        nb[at] = 10 + k
    ix = torch.full((n + 1,), m, dtype=torch.int64, device="cuda")
    ix[0] = 0
    vo = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    lab = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    G._check(G.lib().gpr_batch_cc_noalloc(ix.data_ptr(), nb.data_ptr(), vo.data_ptr(), 1, n, lab.data_ptr(),
                                          C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    want = np.arange(n)
    want[[0, 1, 10, 11, 12, 13, 14, 15]] = 0
    assert np.array_equal(lab.cpu().numpy(), want)


@pytest.mark.parametrize("sizes", [
    [(40, 2)] * 700 + [(60, 8)] * 800,                      # others keep the CUs busy: sparse ones first
    [(40, 2)] * 700 + [(5000, 8)] + [(60, 8)] * 300,        # the largest takes longer than the others
    [(n, 2 if n % 2 else 9) for n in range(2, 1500)],
    [(50, 4)] * 3, [(30, 6)],
])
def test_pinned_labels_in_either_queue_order(sizes):
    G.lib()
    rng = np.random.default_rng(len(sizes))
    voff = np.concatenate(([0], np.cumsum([n for n, _ in sizes]))).astype(np.uint32)
    at = np.repeat(voff[:-1], [n * d // 2 for n, d in sizes])
    size = np.repeat([n for n, _ in sizes], [n * d // 2 for n, d in sizes])
    src, dst = (at + (rng.random(len(at)) * size).astype(np.uint32) for _ in range(2))
    index, nbrs = O.build_csr(int(voff[-1]), src.astype(np.uint32), dst.astype(np.uint32))
    want = O.cc_labels(index, nbrs)
    lab = torch.empty(len(want), dtype=torch.int32, pin_memory=True).numpy().view(np.uint32)
    with G.Batch.from_csr(index, nbrs, voff) as b:
        for _ in range(2):
            lab[:] = 0xFFFFFFFF
            G._check(G.lib().gpr_batch_cc(b.h, lab.ctypes.data_as(C.c_void_p), None))
            assert np.array_equal(lab, want)
            assert np.array_equal(b.cc()[0], want)
