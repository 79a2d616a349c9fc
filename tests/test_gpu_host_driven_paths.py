"""BFS and CC of test-sized graphs by the host-driven loop, which by default
they leave to whole runs (whole_edges)."""
import pytest

pytestmark = pytest.mark.gpu
G = pytest.importorskip("graptor_amd")

from test_gpu_parity import (device, graph, rgraph,                                   # noqa: E402,F401
                             test_bfs_levels_bit_exact, test_bfs_reordered_bit_exact, test_cc_labels_bit_exact,
                             test_cc_push_zero_loops, test_cc_reordered_bit_exact,
                             test_non_symmetric_graph_pull_uses_csc, test_rmat20_bfs_full_size)


@pytest.fixture(autouse=True)
def host_driven():
    G.lib()
    old = G.tune_get("whole_edges")
    G.tune_set("whole_edges", 0)
    yield
    G.tune_set("whole_edges", old)
