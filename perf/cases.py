"""Workloads of the traversal engine: what its users run, over the sizes they run it at.

Each case names an application of the C ABI (the calls that graptor_amd.lib()
binds), a graph and the run's options.  A program keeps the graph handle and
the host buffer that receives the results, and calls the application on them:
that call, results downloaded, is one pass.

Graphs: power-law (RMAT, a=.57 b=.19 c=.19, edge factor 16, folded onto n
vertices where n is no power of two), uniform random (ER), and 2-D grids with
1% random long edges; symmetric ones are relabelled by degree, as the
benchmark does, except the grids.  Sizes run from the test suite's thousand
vertices to the benchmark's RMAT-26.
"""
import ctypes as C
import math

import numpy as np
import torch

import graptor_amd as G

EDGE_FACTOR = 16


def listed():
    return [
        # the smallest call: a BFS on a graph of a few thousand vertices, where launches and read-backs are the time
        {"name": "bfs_rmat_4k", "app": "bfs", "graph": "rmat", "n": 4096},
        # many levels: a mesh with a few long edges, odd sides, from a random vertex
        {"name": "bfs_grid_1021x777", "app": "bfs", "graph": "grid", "n": 1021 * 777, "width": 1021},
        # an ordinary large BFS, few levels, push and pull steps
        {"name": "bfs_rmat_16m", "app": "bfs", "graph": "rmat", "n": 1 << 24},
        # components of a small uniform random graph with isolated vertices, odd size
        {"name": "cc_er_50021", "app": "cc", "graph": "er", "n": 50021},
        # components of a large power-law graph
        {"name": "cc_rmat_32m", "app": "cc", "graph": "rmat", "n": 1 << 25},
        # the benchmark's PageRank: RMAT-26, 20 iterations in FP32
        {"name": "pr_rmat_67m", "app": "pr", "graph": "rmat", "n": 1 << 26, "iters": 20},
        # PageRank of an ordinary small graph, ragged size
        {"name": "pr_rmat_60000", "app": "pr", "graph": "rmat", "n": 60000, "iters": 20},
        # staged precision to convergence on a directed graph: 16-bit contributions first, then FP32
        {"name": "pr_vary_directed_1500007", "app": "pr_vary", "graph": "directed", "n": 1500007, "first": "cfp16"},
        # delta PageRank, the default variant: dense iterations and sparse pushes
        {"name": "apr_rmat_4m", "app": "apr", "graph": "rmat", "n": 1 << 22},
        # core numbers: many levels and rounds of peeling
        {"name": "kcore_rmat_1m", "app": "kcore", "graph": "rmat", "n": 1 << 20},
        # 64 sources in one traversal, the levels of each returned
        {"name": "msbfs_rmat_500000", "app": "msbfs", "graph": "rmat", "n": 500000, "sources": 64},
        # thousands of small graphs in one call
        {"name": "batch_cc_2048", "app": "batch_cc", "graph": "batch", "count": 2048, "nmin": 1024, "nmax": 65536},
    ]


def _log_int(rng, lo, hi):
    """An integer between lo and hi, spread evenly over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    app = rng.choice(("bfs", "bfs", "cc", "cc", "pr", "pr", "pr_vary", "apr", "kcore", "msbfs", "batch_cc"))
    if app == "batch_cc":
        # the allocation-free call on device buffers takes at most 2^21 vertices
        call = rng.choice(("handle", "device"))
        count = _log_int(rng, 16, 2048) if call == "handle" else _log_int(rng, 4, 64)
        nmax = _log_int(rng, 2048, 65536 if call == "handle" else 32768)
        return {"app": app, "graph": "batch", "count": count, "nmin": rng.randint(16, 1024), "nmax": nmax, "call": call}
    case = {"app": app}
    if app == "pr_vary":
        case["graph"] = rng.choice(("directed", "rmat"))
        case["first"] = rng.choice(("cfp16", "bf16", "fp16"))
    elif app in ("bfs", "cc"):
        case["graph"] = rng.choice(("rmat", "rmat", "er", "grid"))
    else:
        case["graph"] = rng.choice(("rmat", "rmat", "er"))
    if case["graph"] == "rmat" and app in ("bfs", "cc", "pr") and rng.random() < 0.25:
        case["n"] = 1 << rng.randint(22, 25)
    elif app == "msbfs":
        case["n"] = _log_int(rng, 1000, 500000)
    elif app == "kcore":
        case["n"] = _log_int(rng, 1000, 1000000)
    else:
        case["n"] = _log_int(rng, 1000, 3000000)
    if case["graph"] == "grid":
        # at most the listed grid's cost: levels grow with the sides
        case["width"] = _log_int(rng, 100, 1000)
        case["n"] = case["width"] * _log_int(rng, 100, 780)
    if app == "bfs" and rng.random() < 0.3:
        case["fusion"] = rng.choice((1, 2))
    if app == "pr":
        case["iters"] = rng.randint(2, 20)
        if rng.random() < 0.4:
            case["format"] = rng.choice(("bf16", "cfp16", "fp16"))
    if app == "msbfs":
        case["sources"] = rng.choice((1, 7, 32, 64))
    return case


# ---- graphs ---------------------------------------------------------------------------------------------------------


def _edges(case, seed):
    """Source and destination of the generated edges, on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n, kind = case["n"], case["graph"]
    if kind in ("rmat", "directed"):
        m = EDGE_FACTOR * n
        scale = max(1, (n - 1).bit_length())
        src = torch.zeros(m, dtype=torch.int64, device="cuda")
        dst = torch.zeros(m, dtype=torch.int64, device="cuda")
        for _ in range(scale):
            r = torch.rand(m, generator=gen, device="cuda")
            src = 2 * src + (r >= 0.76)
            dst = 2 * dst + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
        return src % n, dst % n
    if kind == "er":
        src = torch.randint(0, n, (3 * n,), generator=gen, device="cuda")
        return src, torch.randint(0, n, (3 * n,), generator=gen, device="cuda")
    v = torch.arange(n, device="cuda")
    w, long = case["width"], n // 100
    right, down = v[(v % w) + 1 < w], v[v + w < n]
    far = [torch.randint(0, n, (long,), generator=gen, device="cuda") for _ in range(2)]
    return torch.cat((right, down, far[0])), torch.cat((right + 1, down + w, far[1]))


def _csr(case, seed):
    """The cleaned graph (no self loops, no repeated edges) as offsets and neighbours on the GPU."""
    n = case["n"]
    src, dst = _edges(case, seed)
    keep = src != dst
    key = src[keep] * n + dst[keep]
    if case["graph"] != "directed":
        key = torch.cat((key, dst[keep] * n + src[keep]))
    key = torch.unique(key)
    rows = torch.div(key, n, rounding_mode="floor")
    index = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    index[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
    return index, key - rows * n


def _batch_csr(case, seed):
    """Small graphs side by side: sizes spread over their logarithm (the case's own), every other one power-law (edge
    factor 8), the rest uniform random (mean degree 6); offsets, neighbours and vertex offsets on the host."""
    count, lo, hi = case["count"], case["nmin"], case["nmax"]
    u = np.random.RandomState(count).rand(count)
    nv = np.round(lo * (hi / lo) ** u).astype(np.int64)
    voff = np.concatenate((np.zeros(1, np.int64), np.cumsum(nv)))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    sizes, starts = torch.from_numpy(nv).cuda(), torch.from_numpy(voff[:-1]).cuda()
    even = torch.arange(count, device="cuda") % 2 == 0
    graph = torch.repeat_interleave(torch.arange(count, device="cuda"), torch.where(even, 8 * sizes, 3 * sizes))
    power = even[graph]
    src = torch.zeros_like(graph)
    dst = torch.zeros_like(graph)
    for _ in range(int(hi - 1).bit_length()):
        r = torch.rand(len(graph), generator=gen, device="cuda")
        src = 2 * src + torch.where(power, r >= 0.76, r >= 0.5)
        dst = 2 * dst + torch.where(power, ((r >= 0.57) & (r < 0.76)) | (r >= 0.95), ((r * 4).long() & 1) == 1)
    n = int(voff[-1])
    base, size = starts[graph], sizes[graph]
    src, dst = base + src % size, base + dst % size
    keep = src != dst
    src, dst = src[keep], dst[keep]
    key = torch.unique(torch.cat((src * n + dst, dst * n + src)))
    rows = torch.div(key, n, rounding_mode="floor")
    index = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    index[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
    nbrs = (key - rows * n).to(torch.int32)
    return index.cpu().numpy().view(np.uint64), nbrs.cpu().numpy().view(np.uint32), voff.astype(np.uint32)


def _on_device(case):
    """Whether the graph comes from the engine's own RMAT generator (the large power-law graphs)."""
    return case["graph"] == "rmat" and case["n"] >= 1 << 24


def _graph(case, seed):
    if _on_device(case):
        g = G.Graph.rmat(case["n"].bit_length() - 1, EDGE_FACTOR, 0.57, 0.19, 0.19, seed + 1)
    else:
        index, nbrs = _csr(case, seed)
        host = index.cpu().numpy().astype(np.uint64), nbrs.to(torch.int32).cpu().numpy().view(np.uint32)
        g = G.Graph.from_csr(*host, symmetric=case["graph"] != "directed")
    if case["graph"] in ("rmat", "er"):
        g.reorder()
    return g


# ---- what a program keeps -------------------------------------------------------------------------------------------


def _host(count, dtype):
    """A kept result buffer in pinned host memory."""
    size = max(1, count) * np.dtype(dtype).itemsize
    return torch.empty(size, dtype=torch.uint8, pin_memory=True).numpy().view(dtype)


class State:
    """The handle, the arguments and the result buffers of one case."""

    def __init__(self):
        self.handle = None

    def __del__(self):
        if self.handle is not None:
            self.handle.destroy()


def _stages(pairs):
    return (G.PrStage * len(pairs))(*[G.PrStage(G.CONTRIB_NAMES[f], t) for f, t in pairs])


def prepare(case, seed):
    s = State()
    app = s.app = case["app"]
    rng = np.random.RandomState(seed % (1 << 31))
    if app == "batch_cc":
        s.call = case.get("call", "handle")
        index, nbrs, voff = _batch_csr(case, seed)
        if s.call == "device":
            s.count, s.n = case["count"], int(voff[-1])
            s.index = torch.from_numpy(index.view(np.int64)).cuda()
            s.nbrs = torch.from_numpy(nbrs.view(np.int32)).cuda()
            s.voff = torch.from_numpy(voff.view(np.int32)).cuda()
            s.labels = torch.empty(s.n, dtype=torch.int32, device="cuda")
        else:
            s.handle = G.Batch.from_csr(index, nbrs, voff)
            s.labels = _host(s.handle.n, np.uint32)
        return s
    g = s.handle = _graph(case, seed)
    s.info = G.RunInfo()
    s.opts = G.opts(fusion=case.get("fusion", 0))
    if app == "bfs":
        s.out = _host(g.n, np.uint32)
        s.start = g.highest_degree_vertex() if case["graph"] == "rmat" else int(rng.randint(g.n))
    elif app in ("cc", "kcore"):
        s.out = _host(g.n, np.uint32)
        s.largest = C.c_uint32()
    elif app == "pr":
        s.out = _host(g.n, np.float32)
        s.opts = G.opts(max_iter=case["iters"], tol=0.0)
        s.stages = _stages([(case.get("format", "fp32"), 0.0)])
    elif app == "pr_vary":
        s.out = _host(g.n, np.float32)
        s.stages = _stages([(case["first"], 1e-3), ("fp32", 1e-7)])
    elif app == "apr":
        s.out = _host(g.n, np.float64)
        s.stages = _stages(G.APR_STAGES_2046)
    elif app == "msbfs":
        k = case["sources"]
        s.out = _host(k * g.n, np.uint32).reshape(k, g.n)
        s.src = np.ascontiguousarray(rng.randint(0, g.n, k), np.uint32)
    return s


def _ok(rc):
    if rc != G.GPR_OK:
        text = C.create_string_buffer(1024)
        G.lib().gpr_last_error(text, len(text))
        raise G.GprError(rc, text.value.decode(errors="replace"))


def run(s):
    L, app = G.lib(), s.app
    if app == "batch_cc":
        if s.call == "device":
            stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
            _ok(L.gpr_batch_cc_noalloc(s.index.data_ptr(), s.nbrs.data_ptr(), s.voff.data_ptr(), s.count, s.n,
                                       s.labels.data_ptr(), stream))
        else:
            _ok(L.gpr_batch_cc(s.handle.h, s.labels.ctypes.data, None))
        return s.labels
    h, o, out, info = s.handle.h, C.byref(s.opts), s.out.ctypes.data, C.byref(s.info)
    if app == "bfs":
        _ok(L.gpr_bfslvl(h, s.start, o, out, info))
    elif app == "cc":
        _ok(L.gpr_ccv(h, o, out, info))
    elif app == "kcore":
        _ok(L.gpr_kcore(h, o, out, C.byref(s.largest), info))
        return s.out, s.largest.value
    elif app in ("pr", "pr_vary"):
        _ok(L.gpr_pr_vary(h, s.stages, len(s.stages), o, out, info))
    elif app == "apr":
        _ok(L.gpr_apr_vary(h, s.stages, len(s.stages), 1e-2, o, out, info))
    elif app == "msbfs":
        _ok(L.gpr_msbfs(h, s.src.ctypes.data, len(s.src), o, out, info))
    return s.out


# ---- the least work -------------------------------------------------------------------------------------------------


def _edge_count(case):
    """About how many directed edges the cleaned graph has."""
    n = case["n"]
    if case["graph"] == "er":
        return 6 * n
    if case["graph"] == "grid":
        return 4.02 * n
    kept = 1 - 0.36 * 2.0 ** (-(math.log2(n) - 10) / 4)   # RMAT's repeated edges, fewer on larger graphs
    return (1 if case["graph"] == "directed" else 2) * EDGE_FACTOR * n * kept


def work(case):
    app = case["app"]
    if app == "batch_cc":
        n = case["count"] * (case["nmax"] - case["nmin"]) / max(1e-9, math.log(case["nmax"] / case["nmin"]))
        return {"bytes": 8 * n + 4 * 10 * n + 4 * n, "flops": 0}
    n, m = case["n"], _edge_count(case)
    graph = 8 * (n + 1) + 4 * m
    if app in ("bfs", "cc"):
        # every vertex's offset, one of its edges, its result: a dense step stops at the first useful edge
        return {"bytes": 16 * n, "flops": 0}
    if app == "kcore":
        return {"bytes": graph + 4 * n, "flops": 0}
    if app == "msbfs":
        return {"bytes": graph + 4 * n * case["sources"], "flops": 0}
    # PageRank: per iteration the graph, the contributions read and the sums written; delta PageRank's dense
    # iterations, and about the iterations that the staged run takes to converge
    iters = {"pr": case.get("iters", 20), "pr_vary": 24, "apr": 5}[app]
    return {"bytes": iters * (graph + 8 * n), "flops": iters * 2 * m}


# ---- exact values ---------------------------------------------------------------------------------------------------


def exact(case, seed):
    """PageRank in FP64; the staged run's limit.  The other outputs are whole numbers, or (delta PageRank) depend on
    which vertices its threshold leaves out."""
    app = case["app"]
    if app not in ("pr", "pr_vary") or _on_device(case):
        return None
    n = case["n"]
    index, nbrs = _csr(case, seed)
    deg = index[1:] - index[:-1]
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"), deg)
    scale = torch.where(deg > 0, 0.85 / deg.clamp(min=1).double(), torch.zeros((), dtype=torch.float64, device="cuda"))
    x = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
    for _ in range(case["iters"] if app == "pr" else 80):
        y = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, nbrs, (x * scale)[rows])
        y += (1.0 - y.sum()) / n
        x = y / y.sum()
    return x
