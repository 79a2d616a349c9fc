// msbfs.hip -- multi-source BFS: up to 64 BFSLVLv runs as the bit lanes of
// one traversal.
//
// Per vertex: seen[v] (bit j: reached from source j), cur[v] (bits that
// reached v in the previous level), nxt[v] (bits arriving this level).  One
// level is
//   push (sparse): for the active list, every edge (u,v) ORs cur[u] & ~seen[v]
//                  into nxt[v] (64-bit atomicOr) -- workgroups take tiles of
//                  consecutive frontier edges as in the single-source push;
//   pull (dense):  every v not yet seen by all sources ORs cur[u] over its
//                  in-edges, stopping once every missing bit has arrived;
//                  a workgroup takes a pull bucket (<= STREAM_ITEMS rows +
//                  edges) or a chunk of a long row, so no wave waits for
//                  one that walks the hubs' rows alone;
// followed by a dense finalize: new = nxt & ~seen, seen |= new, cur = new,
// level[v][j] = level+1 for every bit j of new, and the next active list
// (through LDS queues) with its out-degree sum.  The levels are kept by
// vertex, one row of k words each, and turned into the caller's one row a
// source, in original IDs, at the end.  Direction follows the
// reference's rule on the aggregate frontier (nactv + nacte <= m/20 pushes,
// api.h:150-153).  Each lane's result equals a single-source BFSLVLv run
// (bench/BFSLVLv.C:110-254) from that source.
#include "internal.hpp"
#include "device.hpp"

#include <algorithm>
#include <vector>

namespace gpr {

constexpr int MS_THREADS = 256;
constexpr int MS_TILE = 1024;

__global__ void k_ms_init(uint32_t n, uint32_t k, uint32_t *levels, uint64_t *seen, uint64_t *cur, uint64_t *nxt) {
    const uint64_t total = (uint64_t)k * n;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < total; i += (uint64_t)gridDim.x * blockDim.x)
        levels[i] = n + 1;
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
        seen[v] = 0;
        cur[v] = 0;
        nxt[v] = 0;
    }
}

// lane j: source j (k <= 64); two sources may be the same vertex
__global__ void __launch_bounds__(64)
k_ms_sources(const uint32_t *__restrict__ src, uint32_t k, uint32_t *levels, uint64_t *seen, uint64_t *cur) {
    const uint32_t j = threadIdx.x;
    if (j >= k) return;
    const uint32_t s = src[j];
    atomicOr((unsigned long long *)&seen[s], 1ull << j);
    atomicOr((unsigned long long *)&cur[s], 1ull << j);
    levels[(uint64_t)s * k + j] = 0;
}

// push over the active list (degree prefix in pos/btot as for the
// single-source push)
__global__ void __launch_bounds__(MS_THREADS)
k_ms_push(const uint32_t *__restrict__ flist, uint32_t kf, const uint64_t *__restrict__ pos,
          const uint64_t *__restrict__ btot, uint64_t E, const uint64_t *__restrict__ index,
          const uint32_t *__restrict__ nbrs, const uint64_t *__restrict__ cur, const uint64_t *__restrict__ seen,
          uint64_t *nxt) {
    __shared__ uint64_t s_pos[MS_TILE + 1];
    __shared__ uint32_t s_v[MS_TILE + 1];
    __shared__ uint32_t s_i0, s_cnt;
    const uint64_t ntiles = (E + MS_TILE - 1) / MS_TILE;
    for (uint64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const uint64_t e0 = t * MS_TILE, e1 = min(E, e0 + MS_TILE);
        if (threadIdx.x < 64) {
            // the tile's first and last sources, by one wave's 64-way search
            const uint32_t i0 = wave_ub_pos(pos, btot, kf, e0, 0u) - 1;
            const uint32_t i1 = wave_ub_pos(pos, btot, kf, e1 - 1, i0 + 1);
            if (threadIdx.x == 0) {
                s_i0 = i0;
                s_cnt = i1 - i0;
            }
        }
        __syncthreads();
        const uint32_t i0 = s_i0, cnt = s_cnt;
        const bool in_lds = cnt <= MS_TILE + 1;
        if (in_lds)
            for (uint32_t j = threadIdx.x; j < cnt; j += MS_THREADS) {
                s_pos[j] = pos[i0 + j] + btot[(i0 + j) / SCAN_BLOCK];
                s_v[j] = flist[i0 + j];
            }
        __syncthreads();
        for (uint64_t e = e0 + threadIdx.x; e < e1; e += MS_THREADS) {
            uint32_t j;
            if (in_lds) {
                uint32_t lo = 0, hi = cnt;
                while (lo < hi) {
                    uint32_t mid = (lo + hi) >> 1;
                    if (s_pos[mid] <= e) lo = mid + 1; else hi = mid;
                }
                j = lo - 1;
            } else {
                uint32_t lo = i0, hi = i0 + cnt;
                while (lo < hi) {
                    uint32_t mid = (lo + hi) >> 1;
                    if (pos[mid] + btot[mid / SCAN_BLOCK] <= e) lo = mid + 1; else hi = mid;
                }
                j = lo - 1 - i0;
            }
            const uint32_t s = in_lds ? s_v[j] : flist[i0 + j];
            const uint64_t ps = in_lds ? s_pos[j] : pos[i0 + j] + btot[(i0 + j) / SCAN_BLOCK];
            const uint32_t d = nbrs[index[s] + (e - ps)];
            const uint64_t bits = cur[s] & ~seen[d];
            if (bits && (nxt[d] & bits) != bits) atomicOr((unsigned long long *)&nxt[d], bits);
        }
        __syncthreads();
    }
}

// Pull, one workgroup per pull bucket or per chunk of a long row (both from
// the graph's CSC partition).  Bound by the gathers of cur[] (8 B at random;
// they stay in the L2 up to about 500K vertices).  In a bucket: rows up to
// MS_LIGHT in-edges one lane each, MS_PU gathers in flight; longer ones go to
// an LDS queue and are taken by 16 lanes each, 16 * MS_PU edges a step.
// Every row stops once its missing bits have arrived; slots past a row's end
// gather its first neighbour again, which changes no OR.  A long row's
// chunks OR into nxt[row] and stop as well when the row is complete there.
// The split it replaces (a wave per 64 rows, the wave walking their longer
// rows in turn) left the 64 largest hubs to one wave: 6.2 ms a dense level
// on a relabelled 500K-vertex, 15M-edge RMAT graph, 0.06 ms like this.
constexpr int MS_PU = 4;
constexpr uint32_t MS_LIGHT = 32;
constexpr int MS_SUB = 16;   // lanes of a queued row
constexpr uint32_t MS_QCAP = (STREAM_ITEMS + LONG_DEG) / (MS_LIGHT + 1) + 1;

template <int STRIDE>
__device__ __forceinline__ uint64_t ms_gather(const uint32_t *__restrict__ cnbrs, const uint64_t *__restrict__ cur,
                                              uint64_t e, uint64_t first, uint64_t end) {
    uint32_t s[MS_PU];
#pragma unroll
    for (int u = 0; u < MS_PU; ++u) s[u] = cnbrs[e + u * STRIDE < end ? e + u * STRIDE : first];
    uint64_t v = 0;
#pragma unroll
    for (int u = 0; u < MS_PU; ++u) v |= cur[s[u]];
    return v;
}

__global__ void __launch_bounds__(MS_THREADS)
k_ms_pull(uint32_t nbuckets, const uint32_t *__restrict__ bucket, const uint64_t *__restrict__ cindex,
          const uint32_t *__restrict__ cnbrs, const uint32_t *__restrict__ long_rows,
          const uint32_t *__restrict__ long_base, uint32_t nlong, const uint64_t *__restrict__ cur,
          const uint64_t *__restrict__ seen, uint64_t full, uint64_t *nxt) {
    __shared__ uint32_t q[MS_QCAP];
    __shared__ uint32_t qn;
    if (blockIdx.x >= nbuckets) {
        // one chunk of a long row
        const uint32_t c = blockIdx.x - nbuckets;
        uint32_t lo = 0, hi = nlong;   // the row whose chunks c is among
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (long_base[mid] <= c) lo = mid + 1; else hi = mid;
        }
        const uint32_t row = long_rows[lo - 1];
        const uint64_t ms = full & ~seen[row];
        if (!ms) return;
        const uint64_t cb = cindex[row] + (uint64_t)(c - long_base[lo - 1]) * LONG_CHUNK;
        const uint64_t re = cindex[row + 1], ce = cb + LONG_CHUNK < re ? cb + LONG_CHUNK : re;
        uint64_t a = 0;
        for (uint64_t base = cb + (threadIdx.x & ~63u) * MS_PU; base < ce; base += MS_THREADS * MS_PU) {
            uint64_t v = ms_gather<64>(cnbrs, cur, base + lane(), cb, ce);
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v |= __shfl_xor(v, o, 64);
            a |= v;
            const uint64_t have = __hip_atomic_load(&nxt[row], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (((a | have) & ms) == ms) break;
        }
        if (lane() == 0 && (a & ms)) atomicOr((unsigned long long *)&nxt[row], (unsigned long long)(a & ms));
        return;
    }
    if (threadIdx.x == 0) qn = 0;
    __syncthreads();
    const uint32_t r0 = bucket[blockIdx.x], r1 = bucket[blockIdx.x + 1];
    for (uint32_t r = r0 + threadIdx.x; r < r1; r += MS_THREADS) {
        const uint64_t ms = full & ~seen[r];
        if (!ms) continue;
        const uint64_t beg = cindex[r], end = cindex[r + 1];
        if (end - beg > LONG_DEG) continue;   // by its chunks
        if (end - beg > MS_LIGHT) {
            q[atomicAdd(&qn, 1u)] = r;
            continue;
        }
        uint64_t a = 0;
        for (uint64_t e = beg; e < end && (a & ms) != ms; e += MS_PU) a |= ms_gather<1>(cnbrs, cur, e, beg, end);
        if (a & ms) nxt[r] = a & ms;
    }
    __syncthreads();
    const uint32_t cnt = qn, sl = threadIdx.x % MS_SUB;
    for (uint32_t i = threadIdx.x / MS_SUB; i < cnt; i += MS_THREADS / MS_SUB) {
        const uint32_t r = q[i];
        const uint64_t ms = full & ~seen[r];
        const uint64_t beg = cindex[r], end = cindex[r + 1];
        uint64_t a = 0;
        for (uint64_t base = beg; base < end && (a & ms) != ms; base += MS_SUB * MS_PU) {
            uint64_t v = ms_gather<MS_SUB>(cnbrs, cur, base + sl, beg, end);
#pragma unroll
            for (int o = MS_SUB / 2; o > 0; o >>= 1) v |= __shfl_xor(v, o, MS_SUB);
            a |= v;
        }
        if (sl == 0 && (a & ms)) nxt[r] = a & ms;
    }
}

// Finalize a level: levels of the new bits, seen/cur update, next active
// list with its out-degree sum.  Bound by the streams (32 B a vertex) and
// the levels written: a vertex's row is one store of the wave, lane j for
// source j, so each row is written in whole cache lines (one lane per vertex
// with a store per bit: 66 us a dense level at 500K vertices and 64 sources,
// with an atomic a wave on the list position; 28 us like this).
constexpr uint32_t MS_LQ = 512;   // LDS queue entries per wave
__global__ void __launch_bounds__(MS_THREADS)
k_ms_finalize(uint32_t n, uint32_t k, uint32_t level, uint32_t *levels, uint64_t *seen, uint64_t *cur, uint64_t *nxt,
              const uint32_t *__restrict__ deg, uint32_t *list, DevCounters *ctr) {
    __shared__ uint64_t red[MS_THREADS / 64];
    __shared__ uint32_t s_q[MS_THREADS / 64 * MS_LQ];
    __shared__ uint32_t s_c[MS_THREADS / 64], s_base;
    uint64_t my_e = 0;
    const uint32_t ngroups = (n + 63) / 64;
    const uint32_t wid = (blockIdx.x * MS_THREADS + threadIdx.x) / 64, nw = gridDim.x * (MS_THREADS / 64);
    const unsigned ln = lane(), w = threadIdx.x / 64;
    WaveQueue wq{s_q + w * MS_LQ, MS_LQ, 0};
    for (uint32_t grp = wid; grp < ngroups; grp += nw) {
        const uint32_t v = grp * 64 + ln;
        uint64_t nb = 0;
        if (v < n) {
            const uint64_t x = nxt[v];
            if (x) {
                const uint64_t sv = seen[v];
                nb = x & ~sv;
                nxt[v] = 0;
                if (nb) {
                    seen[v] = sv | nb;
                    my_e += deg[v];
                }
            }
            cur[v] = nb;
        }
        const uint64_t word = __ballot(nb != 0);
        for (uint64_t t = word; t; t &= t - 1) {
            const int L = __ffsll((long long)t) - 1;
            const uint64_t b = __shfl(nb, L, 64);
            if ((b >> ln) & 1ull) levels[(uint64_t)(grp * 64 + L) * k + ln] = level + 1;
        }
        wq.push(nb != 0, word, v, list, &ctr->listpos);
    }
    // the waves' remaining queues in one append per workgroup
    if (ln == 0) s_c[w] = wq.cnt;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int j = 0; j < MS_THREADS / 64; ++j) t += s_c[j];
        s_base = t ? atomicAdd(&ctr->listpos, t) : 0u;
    }
    __syncthreads();
    uint32_t off = s_base;
    for (unsigned j = 0; j < w; ++j) off += s_c[j];
    for (uint32_t j = ln; j < wq.cnt; j += 64) list[off + j] = wq.q[j];
    const uint64_t te = block_sum(my_e, red);
    if (threadIdx.x == 0 && te) atomicAdd(&ctr_stripe(ctr)->nacte, (unsigned long long)te);
}

// edges traversed: sum over sources of the out-degrees of reached vertices
__global__ void __launch_bounds__(256)
k_ms_edges(uint32_t n, const uint64_t *__restrict__ seen, const uint32_t *__restrict__ deg, DevCounters *ctr) {
    __shared__ uint64_t red[4];
    uint64_t s = 0;
    for (uint32_t v = blockIdx.x * 256 + threadIdx.x; v < n; v += gridDim.x * 256)
        s += (uint64_t)__popcll(seen[v]) * deg[v];
    s = block_sum(s, red);
    if (threadIdx.x == 0 && s) atomicAdd(&ctr_stripe(ctr)->edges, (unsigned long long)s);
}

// Sources [j0, j0 + js) of the levels as one row of n a source, in original
// IDs: a workgroup turns the rows of MS_OUT_V vertices through LDS, so reads
// are runs of js words and writes runs of MS_OUT_V, whatever the vertex
// order (reading a row a source and scattering it took 216 us at 500K
// vertices and 64 sources, this 93 us).
constexpr uint32_t MS_OUT_V = 64, MS_OUT_J = 16;
__global__ void __launch_bounds__(256)
k_ms_out(const uint32_t *__restrict__ levels, const uint32_t *__restrict__ perm, uint32_t n, uint32_t k, uint32_t j0,
         uint32_t js, uint32_t *dst) {
    __shared__ uint32_t t[MS_OUT_V][MS_OUT_J + 1];
    const uint32_t o0 = blockIdx.x * MS_OUT_V;
    for (uint32_t i = threadIdx.x / MS_OUT_J, j = threadIdx.x % MS_OUT_J; i < MS_OUT_V; i += 256 / MS_OUT_J) {
        const uint32_t o = o0 + i;
        if (o < n && j < js) t[i][j] = levels[(uint64_t)(perm ? perm[o] : o) * k + j0 + j];
    }
    __syncthreads();
    const uint32_t o = o0 + threadIdx.x % MS_OUT_V;
    if (o < n)
        for (uint32_t j = threadIdx.x / MS_OUT_V; j < js; j += 256 / MS_OUT_V)
            dst[(uint64_t)j * n + o] = t[threadIdx.x % MS_OUT_V][j];
}

int scan_frontier_degrees(gpr_graph *g, const uint32_t *list, uint32_t k);

} // namespace gpr

using namespace gpr;

extern "C" int gpr_msbfs(gpr_graph *g, const uint32_t *sources, int k, const gpr_run_opts *opts, uint32_t *levels,
                         gpr_run_info *info) {
    if (!g || !sources || k <= 0 || k > 64) {
        set_error("msbfs: need 1..64 sources");
        return GPR_E_INVAL;
    }
    const uint32_t n = g->n;
    for (int j = 0; j < k; ++j) GPR_REQUIRE(sources[j] < n, "msbfs: source %u out of range", sources[j]);
    const int dir_opt = opts ? opts->direction : GPR_DIR_AUTO;
    const float pct = opts ? opts->threshold_pct : 0.f;   // 0: BFSLVLv's default_threshold
    uint32_t *lev = nullptr, *src = nullptr, *list[2] = {nullptr, nullptr};
    uint64_t *seen = nullptr, *cur = nullptr, *nxt = nullptr;
    int r = GPR_OK;
    gpr_run_info inf = {};
    struct { void *p; size_t bytes; } used[8];
    int nused = 0;
    auto take = [&](void **p, size_t bytes, const char *what) {
        const int e = g->pool->take(p, bytes, what);
        if (e == GPR_OK) used[nused++] = {*p, bytes};
        return e;
    };
    do {
        if ((r = take((void **)&lev, 4ull * k * n, "msbfs levels"))) break;
        if ((r = take((void **)&seen, 8ull * n, "msbfs seen"))) break;
        if ((r = take((void **)&cur, 8ull * n, "msbfs frontier"))) break;
        if ((r = take((void **)&nxt, 8ull * n, "msbfs next"))) break;
        if ((r = take((void **)&list[0], 4ull * n, "msbfs list"))) break;
        if ((r = take((void **)&list[1], 4ull * n, "msbfs list"))) break;
        if ((r = take((void **)&src, 4ull * k, "msbfs sources"))) break;
        std::vector<uint32_t> s(sources, sources + k);
        std::vector<uint32_t> uniq(s);
        std::sort(uniq.begin(), uniq.end());
        uniq.erase(std::unique(uniq.begin(), uniq.end()), uniq.end());
        if (hipMemcpyAsync(src, s.data(), 4ull * k, hipMemcpyHostToDevice, g->stream) != hipSuccess) { r = GPR_E_HIP; break; }
        if ((r = map_ids(g, src, k, true))) break;
        // the first active list: the distinct sources
        if (hipMemcpyAsync(list[0], uniq.data(), 4ull * uniq.size(), hipMemcpyHostToDevice, g->stream) != hipSuccess) {
            r = GPR_E_HIP;
            break;
        }
        if ((r = map_ids(g, list[0], (uint32_t)uniq.size(), true))) break;
        if (!g->rev0) { (void)hipEventCreate(&g->rev0); (void)hipEventCreate(&g->rev1); }
        (void)hipEventRecord(g->rev0, g->stream);
        hipLaunchKernelGGL(k_ms_init, dim3(grid_for((uint64_t)k * n, 256, 16384)), dim3(256), 0, g->stream, n, (uint32_t)k,
                           lev, seen, cur, nxt);
        hipLaunchKernelGGL(k_ms_sources, dim3(1), dim3(64), 0, g->stream, src, (uint32_t)k, lev, seen, cur);
        // out-degree sum of the sources
        uint64_t nacte = 0;
        if ((r = list_edges(g, list[0], (uint32_t)uniq.size(), &nacte))) break;
        uint32_t nactv = (uint32_t)uniq.size();
        const uint64_t full = k == 64 ? ~0ull : ((1ull << k) - 1);
        int cl = 0;
        uint32_t level = 0;
        while (nactv > 0) {
            const bool sparse = dir_opt == GPR_DIR_PUSH ||
                                (dir_opt != GPR_DIR_PULL && threshold_sparse(pct, nactv, nacte, g->m));
            if (sparse) {
                if ((r = scan_frontier_degrees(g, list[cl], nactv))) break;
                if (nacte)
                    hipLaunchKernelGGL(k_ms_push, dim3(grid_for(nacte, MS_TILE, 8192)), dim3(MS_THREADS), 0, g->stream,
                                       list[cl], nactv, g->scan, g->scan_blk, nacte, g->index, g->nbrs, cur, seen, nxt);
                inf.push_iters++;
            } else {
                hipLaunchKernelGGL(k_ms_pull, dim3(g->nbuckets + g->nlong_chunks), dim3(MS_THREADS), 0, g->stream,
                                   g->nbuckets, g->bucket, g->cindex, g->cnbrs, g->long_rows, g->long_base, g->nlong,
                                   cur, seen, full, nxt);
            }
            if ((r = reset_counters(g))) break;
            hipLaunchKernelGGL(k_ms_finalize, dim3(grid_for((n + 63) / 64, MS_THREADS / 64, 2048)), dim3(MS_THREADS), 0,
                               g->stream, n, (uint32_t)k, level, lev, seen, cur, nxt, g->deg, list[cl ^ 1], g->ctr);
            if (hipGetLastError() != hipSuccess) { r = GPR_E_HIP; break; }
            if ((r = read_counters(g))) break;
            nactv = g->hctr->listpos;
            nacte = g->hctr->nacte;
            cl ^= 1;
            ++level;
            inf.iters++;
        }
        if (r) break;
        (void)hipEventRecord(g->rev1, g->stream);
        (void)hipEventSynchronize(g->rev1);
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, g->rev0, g->rev1);
        inf.ms = ms;
        if ((r = reset_counters(g))) break;
        hipLaunchKernelGGL(k_ms_edges, dim3(grid_for(n, 256, 4096)), dim3(256), 0, g->stream, n, seen, g->deg, g->ctr);
        if ((r = read_counters(g))) break;
        inf.edges = g->hctr->edges;
        if (levels) {
            // MS_OUT_J sources at a time through one staging buffer
            uint32_t *tmp = nullptr;
            if ((r = take((void **)&tmp, 4ull * std::min<uint32_t>(k, MS_OUT_J) * n, "msbfs levels"))) break;
            hipError_t e = hipSuccess;
            for (uint32_t j0 = 0; j0 < (uint32_t)k && e == hipSuccess; j0 += MS_OUT_J) {
                const uint32_t js = std::min<uint32_t>(MS_OUT_J, k - j0);
                hipLaunchKernelGGL(k_ms_out, dim3(grid_for(n, MS_OUT_V)), dim3(256), 0, g->stream, lev, g->perm, n,
                                   (uint32_t)k, j0, js, tmp);
                e = hipMemcpyAsync(levels + (uint64_t)j0 * n, tmp, 4ull * js * n, hipMemcpyDeviceToHost, g->stream);
            }
            if (e == hipSuccess) e = hipStreamSynchronize(g->stream);
            if (e != hipSuccess) { r = GPR_E_HIP; break; }
        }
    } while (0);
    if (r == GPR_E_HIP) set_error("msbfs: HIP error %s", hipGetErrorString(hipGetLastError()));
    while (nused) g->pool->give(used[nused - 1].p, used[nused - 1].bytes), --nused;
    if (r == GPR_OK && info) *info = inf;
    return r;
}
