"""Results that go straight into pinned memory of the caller are those that go
through a copy: aligned or not, whole or part of an allocation, each element
size, vertices relabelled or not."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
G = pytest.importorskip("graptor_amd")
torch = pytest.importorskip("torch")
PAD = 96


@pytest.fixture(scope="module", autouse=True)
def device():
    G.lib()
    yield


def into_pinned(nbytes, shift, call):
    """The nbytes that call(pointer) writes `shift` bytes into a pinned block, checked to be all it writes."""
    t = torch.full((nbytes + 2 * PAD,), 0xA5, dtype=torch.uint8).pin_memory()
    call(C.c_void_p(t.data_ptr() + PAD + shift))
    a = t.numpy()
    assert (a[:PAD + shift] == 0xA5).all() and (a[PAD + shift + nbytes:] == 0xA5).all()
    return a[PAD + shift:PAD + shift + nbytes].copy()


@pytest.mark.parametrize("reorder", [False, True])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8, 9, 1023, 4099, 300007])
def test_properties_and_runs(n, reorder):
    k = np.arange(3 * n, dtype=np.uint64)
    index, nbrs = O.build_csr(n, (k * 7919 % n).astype(np.uint32), (k * k * 31 % n).astype(np.uint32))
    rng = np.random.default_rng(n)
    with G.Graph.from_csr(index, nbrs) as g:
        if reorder:
            g.reorder()
        for dt, np_dt in ((G.U16, np.uint16), (G.U32, np.uint32), (G.U64, np.uint64)):
            p = G.Prop(g, dt)
            want = rng.integers(0, 60000, n).astype(np_dt)
            p.upload(want)
            for shift in (0, np.dtype(np_dt).itemsize):
                got = into_pinned(want.nbytes, shift, lambda d: G._check(G.lib().gpr_prop_download(p.h, d)))
                assert np.array_equal(got.view(np_dt), want)
            p.destroy()
        src = np.zeros(2, np.uint32)
        src[1] = n // 2
        ps = src.ctypes.data_as(C.c_void_p)
        for shift in (0, 4):
            info = G.RunInfo()
            got = into_pinned(8 * n, shift, lambda d: G._check(
                G.lib().gpr_msbfs(g.h, ps, 2, None, d, C.byref(info)))).view(np.uint32).reshape(2, n)
            assert np.array_equal(got, O.msbfs_levels(index, nbrs, src))
            got = into_pinned(4 * n, shift, lambda d: G._check(G.lib().gpr_bfslvl(g.h, 0, None, d, C.byref(info))))
            assert np.array_equal(got.view(np.uint32), O.bfs_levels(index, nbrs, 0))
            for o in (None, G.opts(direction=G.DIR_PULL)):       # a whole run and a driven one
                got = into_pinned(4 * n, shift, lambda d: G._check(
                    G.lib().gpr_ccv(g.h, C.byref(o) if o else None, d, C.byref(info))))
                assert np.array_equal(got.view(np.uint32), O.cc_labels(index, nbrs))
            want = g.bfsv(0)[0]
            got = into_pinned(4 * n, shift, lambda d: G._check(G.lib().gpr_bfsv(g.h, 0, None, d, C.byref(info))))
            check_parents(index, nbrs, got.view(np.uint32), want)


def check_parents(index, nbrs, parent, other):
    """Which parent of a level a vertex gets is a race: the reached set is the same, and each is a neighbour."""
    reached = np.flatnonzero(other < 0x80000000)
    assert np.array_equal(reached, np.flatnonzero(parent < 0x80000000))
    for v in reached[:: max(1, len(reached) // 500)]:
        assert v == 0 or parent[v] in nbrs[index[v]:index[v + 1]]


@pytest.mark.parametrize("shift", [0, 4])
def test_batch_labels(shift):
    index, nbrs, voff = O.batch_graphs(20, 100, 2000, 99)
    want, n = O.cc_labels(index, nbrs), len(index) - 1
    with G.Batch.from_csr(index, nbrs, voff) as b:
        info = G.RunInfo()
        for _ in range(3):      # replays with another destination each, and a copied one in between
            got = into_pinned(4 * n, shift, lambda d: G._check(G.lib().gpr_batch_cc(b.h, d, C.byref(info))))
            assert np.array_equal(got.view(np.uint32), want)
            assert np.array_equal(b.cc()[0], want)


def test_batch_labels_in_link_order():
    """More than 8 graphs a CU, half of them sparse: pinned labels have a queue order of their own."""
    count = 2600
    rng = np.random.default_rng(3)
    nv = rng.integers(2, 40, count)
    voff = np.concatenate([[0], np.cumsum(nv)]).astype(np.uint32)
    src, dst = [], []
    for g in range(count):
        m = int(nv[g]) * (1 if g % 2 else 6)
        src.append(voff[g] + rng.integers(0, nv[g], m))
        dst.append(voff[g] + rng.integers(0, nv[g], m))
    n = int(voff[-1])
    index, nbrs = O.build_csr(n, np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32))
    want = O.cc_labels(index, nbrs)
    with G.Batch.from_csr(index, nbrs, voff) as b:
        info = G.RunInfo()
        for _ in range(3):
            got = into_pinned(4 * n, 0, lambda d: G._check(G.lib().gpr_batch_cc(b.h, d, C.byref(info))))
            assert np.array_equal(got.view(np.uint32), want)
            assert np.array_equal(b.cc()[0], want)
