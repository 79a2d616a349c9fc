"""What a graph's runs keep of device memory is bounded, and given back on request."""
import pytest

pytestmark = pytest.mark.gpu
G = pytest.importorskip("graptor_amd")
torch = pytest.importorskip("torch")
MB = 1 << 20


@pytest.fixture(autouse=True)
def restore():
    G.lib()
    old = G.tune_get("pool_vertex_bytes")
    yield
    G.tune_set("pool_vertex_bytes", old)


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def runs(g):
    g.apr_vary(max_iter=3, download=False)
    g.msbfs([1, 2, 3])
    g.prv(max_iter=2, download=False)
    for direction in (G.DIR_AUTO, G.DIR_PULL):
        g.ccv(download=False, direction=direction)
        g.bfslvl(1, download=False, direction=direction)


def test_kept_memory_is_bounded_and_given_back():
    with G.Graph.rmat(22, 4) as g:
        G.tune_set("pool_vertex_bytes", 0)
        runs(g)                                   # layouts and frontier buffers, which stay with the graph
        none = free_bytes()
        runs(g)
        assert abs(free_bytes() - none) <= 16 * MB, "memory is kept with a bound of 0"
        G.tune_set("pool_vertex_bytes", 32)
        runs(g)
        kept = none - free_bytes()
        assert 16 * MB < kept <= 256 * MB + 16 * MB, kept
        G.tune_set("pool_vertex_bytes", 100)      # 400 MB
        runs(g)
        assert none - free_bytes() <= 100 * g.n + 16 * MB
        G.tune_set("pool_vertex_bytes", 0)
        assert abs(free_bytes() - none) <= 16 * MB, "memory is not given back"
