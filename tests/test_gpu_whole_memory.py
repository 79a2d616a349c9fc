"""Runs that find no device memory: what is refused is reported once, and a
whole run leaves the answer to the host-driven run.  Allocations are refused by
a hipMalloc of the test's own that stands before the runtime's, in a process of
its own."""
import os
import subprocess
import sys

import pytest

import oracle as O

pytestmark = pytest.mark.gpu
pytest.importorskip("graptor_amd")

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
size_t refuse_from = 0, refuse_to = 0;   /* sizes refused: [from, to) */
int refused = 0;
int hipMalloc(void **p, size_t n) {
    static int (*real)(void **, size_t);
    if (!real) real = (int (*)(void **, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), "hipMalloc");
    if (n >= refuse_from && n < refuse_to) { ++refused; n = (size_t)1 << 60; }
    return real(p, n);
}
"""

START = r"""
import ctypes as C, sys
import numpy as np
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)     # before the engine, so that its hipMalloc is this one
import graptor_amd as G
import oracle as O
low, high, refused = (C.c_size_t.in_dll(shim, "refuse_from"), C.c_size_t.in_dll(shim, "refuse_to"),
                      C.c_int.in_dll(shim, "refused"))
index, nbrs = O.rmat_graph(16)
n, m = len(index) - 1, len(nbrs)
levels, labels = O.bfs_levels(index, nbrs, 5), O.cc_labels(index, nbrs)
g = G.Graph.from_csr(index, nbrs).reorder()
"""

REPORTED_ONCE = START + r"""
p = g.prop()
p.upload(np.arange(n, dtype=np.uint32))
low.value, high.value = 1, 1 << 62                 # everything
try:
    g.prop(G.F64)
    raise SystemExit("an allocation of %d bytes was not refused" % (8 * n))
except G.GprError as e:
    assert e.code == G.GPR_E_OOM
p.vertex_map(G.VMAP_FILL, 7)                       # asks HIP for its last error after the launch
high.value = 0
assert (p.download() == 7).all() and np.array_equal(g.ccv()[0], labels)
g.destroy()
print("ok")
"""

HOST_DRIVEN = START + r"""
slices = 8 * (m // 256 + min(n, m // 33) + 64)
low.value, high.value = slices, slices + 1         # a whole BFS's slice lists
lv, info = g.bfslvl(5)
assert refused.value > 0, "the slice lists were not asked for"
assert np.array_equal(lv, levels)
high.value = 0
lv, again = g.bfslvl(5)
assert np.array_equal(lv, levels) and (info.iters, info.edges) == (again.iters, again.edges)
assert np.array_equal(g.ccv()[0], labels)
g.destroy()
print("ok")
"""


@pytest.mark.parametrize("script", [REPORTED_ONCE, HOST_DRIVEN], ids=["reported_once", "host_driven"])
def test_refused_allocations(tmp_path, script):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(so), str(src), "-ldl"], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(O.__file__)))
    r = subprocess.run([sys.executable, "-c", script, str(so)], cwd=root, capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, PYTHONPATH=root))
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout, r.stderr[-2000:])
