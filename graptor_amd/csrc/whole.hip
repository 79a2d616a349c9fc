// whole.hip -- BFSLVLv and CCv of small graphs as whole runs on the device.
//
// A host-driven step costs 25-45 us (its launches, the counts read back),
// whatever the frontier: on a graph of a few million edges that is nearly all
// of a run.  Here the host launches a run and waits once.
//
// BFS (k_wb_level): a launch a level, every level a push, queued ahead of the
// device without waiting for counts: a level reads the list lengths that the
// one before left, block 0 tells the host through pinned memory how far
// it is and when the frontier was empty, and the host keeps WB_AHEAD launches
// queued until then (the launches past the end find empty lists and return).
// No barrier inside a launch, so no launch needs all its blocks resident.
// Rows up to WB_LIGHT edges are one lane's work, or that of up to 8 lanes where
// a level leaves lanes idle (a lane's row is a chain of 2.5 us steps of WB_U
// edges: 93 us instead of 76 on RMAT with 4096 vertices, 214 instead of 166 on
// a random graph of 50021); longer ones are listed as WB_SLICE-edge slices, a
// wave each.  A vertex is discovered by atomicMin on
// the levels, which start at n+1: the one that finds n+1 lists it, so no
// bitmap is needed.  A plain load looks first; levels only fall, so what it
// sees at or below the new level proves that there is nothing to do, however
// stale.  Discovered rows are staged per wave in LDS; a workgroup reserves
// list space once, or when a stage fills.  Block 0 counts what the host-driven
// loop reports: its steps, the steps that its threshold rule would push, and
// the frontiers' edges.
//
// CC (k_uf_*): union-find, larger roots hooked under smaller ones, with path
// halving (the scheme of Jaiganesh and Burtscher, "A high-performance
// connected components implementation for GPUs", HPDC 2018).  A vertex starts
// under its first neighbour if that is smaller.  Where no hub joins most of
// the graph that way, two rounds over the first neighbours lower roots by a
// plain atomicMin and flatten the trees; a join lost there is found again.
// Then every edge is joined, over the CSC's pull buckets and long-row chunks,
// and a last pass flattens.  The root of a component is its smallest internal
// ID, the label that CCv converges to.  Parents only fall and each is an
// ancestor, so a stale read costs time only; a join is a compare-and-swap on
// a root, and a failed one looks for the roots again, which are smaller.
#include "internal.hpp"
#include "device.hpp"
#include "label_fold.hpp"
#include "whole.hpp"

#include <algorithm>
#include <cstring>

namespace gpr {

double stream_time_ms(gpr_graph *g, bool start);
void stream_time_mark(gpr_graph *g);
double stream_time_read_ms(gpr_graph *g);

constexpr int WB_THREADS = 256;
constexpr int WB_WAVES = WB_THREADS / 64;
constexpr uint32_t WB_LIGHT = 32;    // rows up to this length: a lane each
constexpr uint32_t WB_SLICE = 256;   // longer rows: a wave per slice of this many edges
constexpr int WB_U = 4;              // edges per lane in flight
constexpr uint32_t WB_STAGE = 512;   // staged list entries per wave
constexpr uint32_t WB_OWN = 64;      // slices of a row that its lane lists alone (with 8: 133 us, not 110, on RMAT of
                                     // 16384 vertices and 4.5M edges, where most rows have some)
constexpr uint32_t WB_TAGS = 256;    // destinations that a workgroup remembers to have tried (wb_claim)
constexpr int WB_CROWD = 16;         // lanes of a wave that gave one up: the rest look past the caches
static_assert(WB_SLICE == 64 * WB_U, "a slice is one pass of the wave");
// A listed row is its first edge and its length, read with the vertex's
// degree when it is discovered: the next level then starts at the neighbours,
// one dependent load sooner.
constexpr int WB_START_BITS = 26;    // first edge (< 2^26 edges); the length (<= WB_LIGHT) above it
static_assert(WB_LIGHT < 1u << (32 - WB_START_BITS), "a light row in 32 bits");

// Counts of the lists, rotating over three slots: level L reads slot L%3,
// adds to (L+1)%3 and clears (L+2)%3, last read by level L-1.  Vertices and
// edges discovered are striped: one line would take an atomic from every
// workgroup of a wide level.
constexpr unsigned WB_STRIPES = 16;
struct alignas(128) WbStripe {
    unsigned long long nact[3], nedge[3];   // vertices discovered, and their out-edges
};
struct alignas(128) WbCtl {
    unsigned int nlight[3], nheavy[3];      // list lengths
    unsigned long long edges;               // of the frontiers so far
    unsigned int pushes;                    // steps the threshold rule would push
    WbStripe stripe[WB_STRIPES];
};

struct WbLists {
    uint32_t *light[2];
    uint64_t *heavy[2];                   // slices: (first edge << 32) | edges
};

// What one wave discovered and has not listed yet (light rows), and its
// counts of the level.
struct WbFound {
    uint32_t *buf;   // WB_STAGE entries of LDS
    unsigned long long *tag;   // the workgroup's WB_TAGS (wb_claim)
    uint32_t n = 0;  // wave-uniform
    uint32_t act = 0;             // per lane
    unsigned long long edge = 0;  // per lane
};

// Graphs with hubs (rows of more than LONG_DEG in-edges): of the lanes of a
// workgroup that see destination d unset, one tries it, as the others' atomics
// could find nothing any more.  Every wave of a wide level sees a hub unset
// before the first atomic on it lands, and they would queue on its line: 500K
// vertices next to the same 16 took 9.8 ms, 0.21 ms like this (host-driven, by
// a pull: 0.14); 0.43 without the second look of a wave in which many lanes
// had the same destination (WB_CROWD).  Dense RMAT graphs gain too: 65536
// vertices with 6M edges 148 -> 130 us.  A slot holds the last destination
// tried and who tried it; a lane that gives up has read its own destination
// written by another lane later than by itself, and the last such lane keeps
// it.  Without hubs the look costs 2-3% and the launch leaves it out.
__device__ __forceinline__ void wb_claim(bool (&need)[WB_U], const uint32_t (&d)[WB_U], unsigned long long *tag) {
#pragma unroll
    for (int j = 0; j < WB_U; ++j) {
        if (!need[j]) continue;
        unsigned long long *t = tag + d[j] % WB_TAGS;
        if ((uint32_t)(__hip_atomic_load(t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >> 32) == d[j])
            need[j] = false;
        else
            __hip_atomic_store(t, (unsigned long long)d[j] << 32 | (threadIdx.x * WB_U + j), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
    }
#pragma unroll
    for (int j = 0; j < WB_U; ++j) {
        if (!need[j]) continue;
        const unsigned long long t = __hip_atomic_load(tag + d[j] % WB_TAGS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        need[j] = (uint32_t)(t >> 32) != d[j] || (uint32_t)t == threadIdx.x * WB_U + j;
    }
}

// The slice of a row's edges from its k-th on.
__device__ __forceinline__ uint64_t wb_slice(uint32_t first, uint32_t len, uint32_t k) {
    return ((uint64_t)(first + k) << 32) | (len - k < WB_SLICE ? len - k : WB_SLICE);
}

__device__ __forceinline__ void wb_store(uint32_t *list, uint32_t at, const WbFound &f) {
    for (uint32_t i = lane(); i < f.n; i += 64) list[at + i] = f.buf[i];
}

// Discover up to WB_U destinations per lane at level nl.  Wave-uniform.
template <bool HUBS>
__device__ __forceinline__ void wb_relax(const bool (&act)[WB_U], const uint32_t (&d)[WB_U], uint32_t nl,
                                         uint32_t *level, const uint64_t *__restrict__ index,
                                         const uint32_t *__restrict__ deg, const WbLists &L, int nb, WbCtl *ctl,
                                         int nx, WbFound &f) {
    bool need[WB_U];
    bool any = false;
#pragma unroll
    for (int j = 0; j < WB_U; ++j)
        need[j] = act[j] && __hip_atomic_load(&level[d[j]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > nl;
#pragma unroll
    for (int j = 0; j < WB_U; ++j) any |= need[j];
    if (!__ballot(any)) return;
    if constexpr (HUBS) {
        const int tried = __popcll(__ballot(any));
        wb_claim(need, d, f.tag);
        any = false;
#pragma unroll
        for (int j = 0; j < WB_U; ++j) any |= need[j];
        if (tried - __popcll(__ballot(any)) >= WB_CROWD) {
#pragma unroll
            for (int j = 0; j < WB_U; ++j)
                need[j] = need[j] && __hip_atomic_load(&level[d[j]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) > nl;
        }
    }
    uint32_t old[WB_U], dg[WB_U], first[WB_U];
#pragma unroll
    for (int j = 0; j < WB_U; ++j) {
        old[j] = need[j] ? atomicMin(&level[d[j]], nl) : 0u;
        dg[j] = need[j] ? deg[d[j]] : 0u;
        first[j] = need[j] ? (uint32_t)index[d[j]] : 0u;
    }
    uint32_t ch = 0;
#pragma unroll
    for (int j = 0; j < WB_U; ++j) {
        const bool found = need[j] && old[j] > nl;
        if (found) {
            ++f.act;
            f.edge += dg[j];
        }
        dg[j] = found ? dg[j] : 0u;
        const bool light = dg[j] > 0 && dg[j] <= WB_LIGHT;
        const uint64_t word = __ballot(light);
        if (word) {
            if (f.n + 64 > WB_STAGE) {
                __builtin_amdgcn_wave_barrier();
                uint32_t b = 0;
                if (lane() == 0) b = atomicAdd(&ctl->nlight[nx], f.n);
                wb_store(L.light[nb], __builtin_amdgcn_readfirstlane(b), f);
                __builtin_amdgcn_wave_barrier();
                f.n = 0;
            }
            if (light) f.buf[f.n + mbcnt(word)] = first[j] | dg[j] << WB_START_BITS;
            f.n += (uint32_t)__popcll(word);
        }
        if (dg[j] > WB_LIGHT) ch += (dg[j] + WB_SLICE - 1) / WB_SLICE;
    }
    if (!__ballot(ch)) return;
    const uint32_t ih = wave_incl_scan(ch), th = __shfl(ih, 63, 64);
    uint32_t b = 0;
    if (lane() == 0) b = atomicAdd(&ctl->nheavy[nx], th);
    b = __builtin_amdgcn_readfirstlane(b) + (ih - ch);
    // A row's lane lists up to WB_OWN slices; more of them the wave lists, 64
    // at a time (by one lane the slices of a row of 4M edges took 500 us).
#pragma unroll
    for (int j = 0; j < WB_U; ++j) {
        const uint32_t sl = dg[j] > WB_LIGHT ? (dg[j] + WB_SLICE - 1) / WB_SLICE : 0u;
        if (sl <= WB_OWN)
            for (uint32_t k = 0; k < sl; ++k) L.heavy[nb][b + k] = wb_slice(first[j], dg[j], k * WB_SLICE);
        for (uint64_t t = __ballot(sl > WB_OWN); t; t &= t - 1) {
            const int o = __ffsll((long long)t) - 1;
            const uint32_t of = __shfl(first[j], o, 64), od = __shfl(dg[j], o, 64), ob = __shfl(b, o, 64);
            for (uint32_t k = lane(); k * WB_SLICE < od; k += 64) L.heavy[nb][ob + k] = wb_slice(of, od, k * WB_SLICE);
        }
        b += sl;
    }
}

// The threshold rule (threshold_sparse): integer nactv + nacte <= limit, or
// with frac its float and double roundings against rhs.
struct WbRule {
    unsigned long long limit;
    double rhs;
    int frac;
};

// What block 0 tells the host (pinned memory).
constexpr unsigned WB_EVERY = 4;
struct alignas(128) WbHost {
    unsigned int level;             // levels begun, every WB_EVERY of them
    unsigned int done;              // 1: the frontier was empty; the fields below are final
    unsigned int steps, pushes;
    unsigned long long edges;
};
static_assert(sizeof(WbHost) == WHOLE_LINE, "the graph keeps one line for it");

// Levels n+1 but for the start's 0, the start's row as the first frontier,
// the counts.
__global__ void __launch_bounds__(WB_THREADS)
k_wb_init(uint32_t n, const uint64_t *__restrict__ index, const uint32_t *__restrict__ deg,
          const uint32_t *__restrict__ perm, uint32_t start, uint32_t *level, WbLists L, WbCtl *ctl) {
    const uint32_t s = perm ? perm[start] : start;
    for (uint32_t v = blockIdx.x * WB_THREADS + threadIdx.x; v < n; v += gridDim.x * WB_THREADS)
        level[v] = v == s ? 0u : n + 1;
    if (blockIdx.x != 0) return;
    const uint32_t ds = deg[s], es = (uint32_t)index[s];
    const uint32_t sl = ds > WB_LIGHT ? (ds + WB_SLICE - 1) / WB_SLICE : 0u;
    for (uint32_t k = threadIdx.x; k < sl; k += WB_THREADS) L.heavy[0][k] = wb_slice(es, ds, k * WB_SLICE);
    unsigned int *w = (unsigned int *)ctl;
    for (unsigned i = threadIdx.x; i < sizeof(WbCtl) / 4; i += WB_THREADS) w[i] = 0;
    __syncthreads();
    if (threadIdx.x == 0) {
        if (ds && !sl) L.light[0][0] = es | ds << WB_START_BITS;
        ctl->nlight[0] = ds && !sl;
        ctl->nheavy[0] = sl;
        ctl->stripe[0].nact[0] = 1;
        ctl->stripe[0].nedge[0] = ds;
    }
}

template <bool HUBS>
__global__ void __launch_bounds__(WB_THREADS)
k_wb_level(uint32_t n, uint32_t lvl, const uint64_t *__restrict__ index, const uint32_t *__restrict__ nbrs,
           const uint32_t *__restrict__ deg, uint32_t *level, WbLists L, WbCtl *ctl, WbRule rule, WbHost *h,
           uint32_t sub_max) {
    __shared__ uint32_t s_stage[WB_WAVES * WB_STAGE];
    __shared__ uint32_t s_n[WB_WAVES], s_act[WB_WAVES], s_base[WB_WAVES];
    __shared__ unsigned long long s_edge[WB_WAVES], s_tag[WB_TAGS];
    const unsigned ln = lane(), wv = threadIdx.x / 64;
    const uint32_t W = gridDim.x * WB_WAVES;
    // wave rank interleaved over the blocks: a small level lands on many CUs
    const uint32_t w = wv * gridDim.x + blockIdx.x;
    const int c = lvl % 3, nx = (lvl + 1) % 3, stale = (lvl + 2) % 3, cb = lvl & 1, nb = cb ^ 1;
    // the wave's first rows are loaded beside the lengths that say whether
    // they are there (a list holds n rows)
    uint32_t row = L.light[cb][min(w * 64 + ln, n - 1)];
    const uint32_t nL = ctl->nlight[c], nH = ctl->nheavy[c];
    if (blockIdx.x == 0) {
        unsigned long long na = 0, ne = 0;
        if (threadIdx.x < WB_STRIPES) {
            WbStripe &st = ctl->stripe[threadIdx.x];
            na = st.nact[c];
            ne = st.nedge[c];
            st.nact[stale] = 0;
            st.nedge[stale] = 0;
        }
        if (threadIdx.x < 64) {
            na = wave_sum(na);
            ne = wave_sum(ne);
        }
        if (threadIdx.x == 0) {
            ctl->nlight[stale] = 0;
            ctl->nheavy[stale] = 0;
            if (na) {
                ctl->edges += ne;
                ctl->pushes += rule.frac ? (double)(float)(na + ne) <= rule.rhs : na + ne <= rule.limit;
            } else if (!h->done) {
                h->steps = lvl;
                h->pushes = ctl->pushes;
                h->edges = ctl->edges;
                __hip_atomic_store(&h->done, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
            }
            if ((lvl + 1) % WB_EVERY == 0)
                __hip_atomic_store(&h->level, lvl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    if constexpr (HUBS) {
        for (uint32_t i = threadIdx.x; i < WB_TAGS; i += WB_THREADS) s_tag[i] = ~0ull;
        __syncthreads();
    }
    // 2^lg lanes a row while there are lanes to spare (up to sub_max)
    uint32_t lg = 0;
    while ((1u << lg) < sub_max && ((uint64_t)nL << (lg + 1)) <= (uint64_t)W * 64) ++lg;
    const uint32_t sub = 1u << lg, rows = 64 >> lg;
    WbFound f{&s_stage[wv * WB_STAGE], s_tag};
    for (uint32_t base = w * rows; base < nL; base += W * rows) {
        const uint32_t i = base + (ln >> lg);
        if (lg || base != w * 64) row = L.light[cb][min(i, n - 1)];
        uint32_t e = 0, e1 = 0;
        if (i < nL) {
            e = row & ((1u << WB_START_BITS) - 1);
            e1 = e + (row >> WB_START_BITS);
            e += ln & (sub - 1);
        }
        while (__ballot(e < e1)) {
            bool act[WB_U];
            uint32_t d[WB_U];
#pragma unroll
            for (int j = 0; j < WB_U; ++j) {
                act[j] = e + (j << lg) < e1;
                d[j] = act[j] ? nbrs[e + (j << lg)] : 0u;
            }
            e += WB_U << lg;    // < 2^26 + 64: no wrap
            wb_relax<HUBS>(act, d, lvl + 1, level, index, deg, L, nb, ctl, nx, f);
        }
    }
    for (uint32_t j = W - 1 - w; j < nH; j += W) {
        const uint64_t ent = L.heavy[cb][j];
        const uint32_t e0 = (uint32_t)(ent >> 32), len = (uint32_t)ent;
        bool act[WB_U];
        uint32_t d[WB_U];
#pragma unroll
        for (int k = 0; k < WB_U; ++k) {
            act[k] = ln + 64 * k < len;
            d[k] = act[k] ? nbrs[e0 + ln + 64 * k] : 0u;
        }
        wb_relax<HUBS>(act, d, lvl + 1, level, index, deg, L, nb, ctl, nx, f);
    }
    // the block's stages and counts, with one reservation
    const uint32_t ta = wave_sum(f.act);
    const unsigned long long te = wave_sum(f.edge);
    if (ln == 0) {
        s_n[wv] = f.n;
        s_act[wv] = ta;
        s_edge[wv] = te;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t tn = 0, a = 0;
        unsigned long long e = 0;
        for (int i = 0; i < WB_WAVES; ++i) {
            s_base[i] = tn;
            tn += s_n[i];
            a += s_act[i];
            e += s_edge[i];
        }
        if (a) {
            WbStripe &st = ctl->stripe[blockIdx.x % WB_STRIPES];
            const uint32_t b = tn ? atomicAdd(&ctl->nlight[nx], tn) : 0u;
            atomicAdd(&st.nact[nx], (unsigned long long)a);
            atomicAdd(&st.nedge[nx], e);
            for (int i = 0; i < WB_WAVES; ++i) s_base[i] += b;
        }
    }
    __syncthreads();
    wb_store(L.light[nb], s_base[wv], f);
}

// Results in original IDs, in order (they may go to host memory).
__global__ void __launch_bounds__(WB_THREADS)
k_wb_out(uint32_t n, const uint32_t *__restrict__ level, const uint32_t *__restrict__ perm, uint32_t *out) {
    for (uint32_t o = blockIdx.x * WB_THREADS + threadIdx.x; o < n; o += gridDim.x * WB_THREADS)
        out[o] = level[perm ? perm[o] : o];
}

// ---- union-find CC ------------------------------------------------------------
constexpr int UF_THREADS = 256;
constexpr uint32_t UF_LIGHT = 32;
constexpr int UF_SUB = 16;
constexpr uint32_t UF_QCAP = (STREAM_ITEMS + LONG_DEG) / (UF_LIGHT + 1) + 1;

template <int SCOPE> __device__ __forceinline__ uint32_t uf_get(const uint32_t *parent, uint32_t v) {
    return __hip_atomic_load(&parent[v], __ATOMIC_RELAXED, SCOPE);
}
// The root above v, halving the path on the way.
template <int SCOPE> __device__ __forceinline__ uint32_t uf_root(uint32_t *parent, uint32_t v) {
    uint32_t p = uf_get<SCOPE>(parent, v);
    while (p != v) {
        const uint32_t q = uf_get<SCOPE>(parent, p);
        if (q == p) return p;
        __hip_atomic_store(&parent[v], q, __ATOMIC_RELAXED, SCOPE);
        v = p;
        p = q;
    }
    return v;
}
// Join the components of a and b.  The first look goes through the caches,
// which hold nearly every answer on a flattened forest; only after a failed
// swap does it read past them (reads of one hot root from every edge would
// queue).
__device__ __forceinline__ void uf_join(uint32_t *parent, uint32_t a, uint32_t b) {
    a = uf_root<__HIP_MEMORY_SCOPE_WORKGROUP>(parent, a);
    b = uf_root<__HIP_MEMORY_SCOPE_WORKGROUP>(parent, b);
    while (a != b) {
        const uint32_t hi = a > b ? a : b, lo = a > b ? b : a;
        const uint32_t old = atomicCAS(&parent[hi], hi, lo);
        if (old == hi) return;
        a = uf_root<__HIP_MEMORY_SCOPE_AGENT>(parent, old);   // hi was hooked already, under old < hi
        b = uf_root<__HIP_MEMORY_SCOPE_AGENT>(parent, lo);
    }
}

__global__ void __launch_bounds__(UF_THREADS)
k_uf_init(uint32_t n, const uint64_t *__restrict__ index, const uint32_t *__restrict__ nbrs, uint32_t *parent,
          uint32_t *minorig, unsigned long long *began) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *began = wall_clock64();
    for (uint32_t v = blockIdx.x * UF_THREADS + threadIdx.x; v < n; v += gridDim.x * UF_THREADS) {
        const uint64_t b = index[v];
        uint32_t p = v;
        if (b < index[v + 1]) p = min(v, nbrs[b]);
        parent[v] = p;
        if (minorig) minorig[v] = 0xffffffffu;
    }
}

// One round over the first UF_FIRST_NBRS neighbours: the larger of two roots
// goes under the smaller by atomicMin, without a second try.  A root that was
// hooked in between may lose that hook to a smaller one; k_uf_link sees every
// edge again.  On a random graph of 500K vertices and 3M edges joining every
// edge at once took 1.5-2.5 ms, most swaps failing on roots that had just
// been hooked; after two rounds the whole run takes 0.3-0.4 ms.
constexpr uint64_t UF_FIRST_NBRS = 4;
constexpr int UF_ROUNDS = 2;
constexpr uint32_t UF_TAGS = 256;
__global__ void __launch_bounds__(UF_THREADS)
k_uf_round(uint32_t n, const uint64_t *__restrict__ index, const uint32_t *__restrict__ nbrs, uint32_t *parent) {
    constexpr int WG = __HIP_MEMORY_SCOPE_WORKGROUP;
    // the pairs that this workgroup tried last, and who did (as wb_claim; a
    // join given up for nothing is found again): two hubs next to the same 2M
    // vertices took 1.5 ms of atomics on their lines, 10 us like this
    __shared__ unsigned long long s_pair[UF_TAGS];
    __shared__ uint32_t s_who[UF_TAGS];
    for (uint32_t i = threadIdx.x; i < UF_TAGS; i += UF_THREADS) s_pair[i] = ~0ull;
    __syncthreads();
    for (uint32_t v = blockIdx.x * UF_THREADS + threadIdx.x; v < n; v += gridDim.x * UF_THREADS) {
        const uint64_t b = index[v], e = min(index[v + 1], b + UF_FIRST_NBRS);
        const uint32_t a = uf_get<WG>(parent, v);
        for (uint64_t j = b; j < e; ++j) {
            const uint32_t c = uf_get<WG>(parent, nbrs[j]);
            const uint32_t hi = a > c ? a : c, lo = a > c ? c : a;
            if (hi == lo || uf_get<WG>(parent, hi) <= lo) continue;
            const unsigned long long pair = (unsigned long long)hi << 32 | lo;
            unsigned long long *t = s_pair + hi % UF_TAGS;
            uint32_t *w = s_who + hi % UF_TAGS;
            if (__hip_atomic_load(t, __ATOMIC_RELAXED, WG) == pair) continue;
            __hip_atomic_store(t, pair, __ATOMIC_RELAXED, WG);
            __hip_atomic_store(w, threadIdx.x, __ATOMIC_RELAXED, WG);
            if (__hip_atomic_load(t, __ATOMIC_RELAXED, WG) == pair && __hip_atomic_load(w, __ATOMIC_RELAXED, WG) != threadIdx.x)
                continue;
            atomicMin(&parent[hi], lo);
        }
    }
}

// Every edge once, from its larger endpoint; the split of rows as in the
// 64-source pull: lanes, 16-lane groups, chunks of long rows.
__global__ void __launch_bounds__(UF_THREADS)
k_uf_link(uint32_t nbuckets, const uint32_t *__restrict__ bucket, const uint64_t *__restrict__ index,
          const uint32_t *__restrict__ nbrs, const uint32_t *__restrict__ long_rows,
          const uint32_t *__restrict__ long_base, uint32_t nlong, uint32_t *parent) {
    __shared__ uint32_t q[UF_QCAP];
    __shared__ uint32_t qn;
    if (blockIdx.x >= nbuckets) {
        const uint32_t c = blockIdx.x - nbuckets;
        uint32_t lo = 0, hi = nlong;   // the row whose chunks c is among
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (long_base[mid] <= c) lo = mid + 1; else hi = mid;
        }
        const uint32_t row = long_rows[lo - 1];
        const uint64_t cb = index[row] + (uint64_t)(c - long_base[lo - 1]) * LONG_CHUNK;
        const uint64_t re = index[row + 1], ce = cb + LONG_CHUNK < re ? cb + LONG_CHUNK : re;
        for (uint64_t e = cb + threadIdx.x; e < ce; e += UF_THREADS) {
            const uint32_t u = nbrs[e];
            if (u < row) uf_join(parent, row, u);
        }
        return;
    }
    if (threadIdx.x == 0) qn = 0;
    __syncthreads();
    const uint32_t r0 = bucket[blockIdx.x], r1 = bucket[blockIdx.x + 1];
    for (uint32_t r = r0 + threadIdx.x; r < r1; r += UF_THREADS) {
        const uint64_t beg = index[r], end = index[r + 1];
        if (end - beg > LONG_DEG) continue;   // by its chunks
        if (end - beg > UF_LIGHT) {
            q[atomicAdd(&qn, 1u)] = r;
            continue;
        }
        for (uint64_t e = beg; e < end; ++e) {
            const uint32_t u = nbrs[e];
            if (u < r) uf_join(parent, r, u);
        }
    }
    __syncthreads();
    const uint32_t cnt = qn;
    for (uint32_t i = threadIdx.x / UF_SUB; i < cnt; i += UF_THREADS / UF_SUB) {
        const uint32_t r = q[i];
        const uint64_t end = index[r + 1];
        for (uint64_t e = index[r] + threadIdx.x % UF_SUB; e < end; e += UF_SUB) {
            const uint32_t u = nbrs[e];
            if (u < r) uf_join(parent, r, u);
        }
    }
}

// Every vertex under its root; with minorig, the components' smallest
// original IDs at the roots too.  A launch of its own, so no root is hooked
// meanwhile.  A few parents may still be inner ancestors afterwards: halving
// stores of other threads that come late.
__global__ void __launch_bounds__(LF_THREADS)
k_uf_flatten(uint32_t n, uint32_t *parent, const uint32_t *__restrict__ order, uint32_t *minorig) {
    constexpr int WG = __HIP_MEMORY_SCOPE_WORKGROUP;
    LabelFold f;
    for (uint64_t i = blockIdx.x * (uint64_t)LF_THREADS + threadIdx.x; i < n; i += (uint64_t)gridDim.x * LF_THREADS) {
        const uint32_t r = uf_root<WG>(parent, (uint32_t)i);
        __hip_atomic_store(&parent[i], r, __ATOMIC_RELAXED, WG);
        if (minorig) f.add(minorig, i, r, order[i]);
    }
    if (minorig) f.finish(minorig);
}

// The root above v in a forest at rest: nearly always its parent.
__device__ __forceinline__ uint32_t uf_top(const uint32_t *__restrict__ parent, uint32_t v) {
    uint32_t p = parent[v];
    while (p != v) {
        v = p;
        p = parent[v];
    }
    return v;
}
__global__ void __launch_bounds__(UF_THREADS)
k_uf_out(uint32_t n, const uint32_t *__restrict__ parent, const uint32_t *__restrict__ perm,
         const uint32_t *__restrict__ minorig, uint32_t *out, unsigned long long *ended) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *ended = wall_clock64();
    for (uint32_t o = blockIdx.x * UF_THREADS + threadIdx.x; o < n; o += gridDim.x * UF_THREADS) {
        const uint32_t r = uf_top(parent, perm ? perm[o] : o);
        out[o] = minorig ? minorig[r] : r;
    }
}

// ---- host side ------------------------------------------------------------------
constexpr uint32_t WHOLE_STAGE_V = 1u << 18;   // results up to this many vertices go straight to pinned memory

// The line at whole_edges (2^24): a whole BFS against the host-driven one,
// results downloaded, in us: RMAT 0.1M edges 99 / 190, 1.8M 135 / 236, 7.6M
// 253 / 260, 15M 289 / 361, 31M 458 / 387 (a dense level is cheaper pulled);
// meshes and random graphs, of more levels, gain everywhere (8M edges 1300 /
// 3200 and 593 / 735).  Whole CC gains to twice that: RMAT 0.1M 47 / 230, 7.6M
// 131 / 317, 31M 257 / 457, 128M 1055 / 764; random 18M 1150 / 1840.
// Below these limits too the host-driven run is the better one where its pulls
// save most of the edges, or where a join's random reads leave the L2:
//   BFS with 32 edges a vertex or more, from 2^23 edges and 2^15 vertices on
//   (below, the levels stay in the nearer caches), but for relabelled graphs
//   with hubs.  Whole / host-driven, results left on the device: random
//   graphs, 250000 vertices of 60 edges 383 / 215, 500000 of 32 555 / 343,
//   100000 of 150 198 / 169, 60000 of 250 186 / 159, but 30000 of 500 122 /
//   184, 250000 of 30 283 / 283, 100000 of 60 208 / 211; RMAT 262144 of 55
//   234 / 244 in its own order, relabelled 186 / 264;
//   CC with hubs in their own order, from 2^24 edges and 2^16 vertices on, or
//   3 2^22 edges and 2^20 vertices (a 4 MB L2 of parents).  RMAT, results left
//   on the device: 33M edges on 4M vertices 641 / 386, 31M on 1M 378 / 243, 23M
//   on 0.5M 274 / 224, 19M on 131072 240 / 171, but on 65536 175 / 202; 16.6M on
//   4M 498 / 376, 12.4M on 2M 329 / 314, 15.5M on 0.5M 230 / 225.  Without a hub
//   next to most of the graph it loses: 1000 hubs, each next to 12000 of 200000
//   vertices, 303 / 452.
static bool host_driven_better(const gpr_graph *g, bool cc) {
    if (cc)
        return !g->order && g->nlong && ((g->m > (1u << 24) && g->n > (1u << 16)) ||
                                         (g->m > 3u << 22 && g->n > (1u << 20)));
    return g->m > (1u << 23) && g->n > (1u << 15) && g->m >= 32ull * g->n && !(g->order && g->nlong);
}
bool whole_run(const gpr_graph *g, const gpr_run_opts &o, bool cc) {
    const double limit = std::min(tun().whole_edges * (cc ? 2.0 : 1.0), (double)(1u << WB_START_BITS));
    if ((double)g->m > limit || (double)g->n > limit || g->n == 0 || host_driven_better(g, cc)) return false;
    if (o.direction != GPR_DIR_AUTO || o.out_kind != 0 || o.trace || o.deferred_update || g->prof.on) return false;
    return cc ? o.fusion == 0 && g->symmetric && !(o.threshold_pct > 0.f) : o.fusion <= 0;
}

// A run's device memory: the graph's 8 (n+1) bytes of scan scratch, and blocks
// of its pool, which keeps them for the next run.  Several blocks rather than
// one, as hipMalloc takes 0.3 ms from 2 MB on and little below: the first BFS
// of a fresh handle on 200000 vertices and 5.5M edges takes 210 us, 530 with
// one block, 560 with buffers of its own and staging memory made whatever the
// destination; host-driven 410.  A CC needs no block, but for labels in
// pageable memory: 100 us there, 200 with its own buffers.
struct WholeMem {
    gpr_graph *g;
    struct { void *p; size_t bytes; } used[4];
    int n = 0;
    explicit WholeMem(gpr_graph *gr) : g(gr) {}
    WholeMem(const WholeMem &) = delete;
    ~WholeMem() { while (n) --n, g->pool->give(used[n].p, used[n].bytes); }
    template <class T> int take(T **p, size_t bytes, const char *what) {
        void *q = nullptr;
        GPR_TRY(g->pool->take(&q, bytes, what));
        used[n++] = {q, bytes};
        *p = (T *)q;
        return GPR_OK;
    }
};

// Pinned memory for n results that go to a buffer the device cannot write:
// small graphs', from the second such run on.
static uint32_t *whole_stage(gpr_graph *g) {
    if (g->n > WHOLE_STAGE_V || (!g->wstage && g->wstage_runs++ == 0)) return nullptr;
    if (!g->wstage) {
        void *p = nullptr, *d = nullptr;
        if (hipHostMalloc(&p, 4ull * g->n, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess ||
            hipHostGetDevicePointer(&d, p, 0) != hipSuccess) {
            (void)hipGetLastError();
            if (p) hipHostFree(p);
            return nullptr;
        }
        g->wstage = (uint32_t *)p;
        g->wstage_dev = (uint32_t *)d;
    }
    return g->wstage_dev;
}
// Waits for the stream; the n results at dev (the staging memory or the
// device) into host, when asked for.
static int whole_results(gpr_graph *g, const uint32_t *dev, uint32_t *host, bool direct) {
    const bool staged = !direct && dev == g->wstage_dev;
    if (host && !staged && !direct) GPR_HIP(hipMemcpyAsync(host, dev, 4ull * g->n, hipMemcpyDeviceToHost, g->stream));
    GPR_HIP(hipStreamSynchronize(g->stream));
    if (host && staged) std::memcpy(host, g->wstage, 4ull * g->n);
    return GPR_OK;
}

// Launches queued beyond the last level reported: the host needs about 4 us a
// launch and a small level takes 8; those past the end cost about 3 us each.
// Reporting every level instead of every fourth (a write to the host that
// the launch waits for) took 460 us instead of 434 on 47 levels.
constexpr unsigned WB_AHEAD = 6;
// Blocks of a level's launch: one per WB_BLOCK_EDGES edges of the graph.  With
// 32 at least instead of 128, a random graph of 50021 vertices took 182 us, not
// 166; one of 4096 (RMAT) 87, not 76.
constexpr uint64_t WB_BLOCK_EDGES = 4096;
constexpr uint64_t WB_MIN_BLOCKS = 128;

int whole_bfs(gpr_graph *g, uint32_t start, float threshold_pct, uint32_t *levels, gpr_run_info *info) {
    const uint32_t n = g->n;
    const uint32_t *perm = g->order ? g->perm : nullptr;
    // a level's slices: each row of more than WB_LIGHT edges has one at least
    const uint64_t nheavy = g->m / WB_SLICE + std::min<uint64_t>(n, g->m / (WB_LIGHT + 1)) + 64;
    WholeMem mem(g);
    uint32_t *level = nullptr;
    WbCtl *ctl = nullptr;
    WbLists L = {{(uint32_t *)g->scan, (uint32_t *)g->scan + n}, {nullptr, nullptr}};
    GPR_TRY(mem.take(&level, 4ull * n, "levels"));
    GPR_TRY(mem.take(&L.heavy[0], 8 * nheavy, "whole BFS lists"));
    GPR_TRY(mem.take(&L.heavy[1], 8 * nheavy, "whole BFS lists"));
    GPR_TRY(mem.take(&ctl, sizeof(WbCtl), "whole BFS control"));
    WbRule rule = {g->m / 20, 0.0, 0};
    if (threshold_pct > 0.f) {
        rule.frac = 1;
        rule.rhs = (double)(float)g->m / (100.0 / (double)threshold_pct);
    }
    const unsigned grid = (unsigned)std::min<uint64_t>(1024, std::max<uint64_t>(WB_MIN_BLOCKS, g->m / WB_BLOCK_EDGES));
    // lanes that an average row keeps busy for one step
    uint32_t sub_max = 1;
    while (sub_max * WB_U < WB_LIGHT && (uint64_t)sub_max * WB_U * n < g->m) sub_max *= 2;
    WbHost *const hline = (WbHost *)g->wline;
    volatile WbHost *h = hline;
    h->level = 0;
    h->done = 0;
    stream_time_ms(g, true);
    hipLaunchKernelGGL(k_wb_init, dim3(grid_for(n, WB_THREADS, 1024)), dim3(WB_THREADS), 0, g->stream, n, g->index,
                       g->deg, perm, start, level, L, ctl);
    unsigned launched = 0, polls = 0;
    hipError_t e = hipGetLastError();
    while (!__atomic_load_n(&hline->done, __ATOMIC_ACQUIRE)) {
        if (launched - h->level < WB_AHEAD) {
            hipLaunchKernelGGL(g->nlong ? k_wb_level<true> : k_wb_level<false>, dim3(grid), dim3(WB_THREADS), 0,
                               g->stream, n, launched, g->index, g->nbrs, g->deg, level, L, ctl, rule,
                               (WbHost *)g->wline_dev, sub_max);
            ++launched;
            e = hipGetLastError();
        } else if (++polls % 4096 == 0) {
            // a stream that failed would never report a level
            e = hipStreamQuery(g->stream);
            if (e == hipErrorNotReady) {
                e = hipSuccess;
                (void)hipGetLastError();
            }
        }
        if (e != hipSuccess) {
            // the queued levels still write the progress line, which the next
            // run of the handle resets
            (void)hipStreamSynchronize(g->stream);
            GPR_HIP(e);
        }
    }
    stream_time_mark(g);
    bool copy_only = false;
    uint32_t *const target = (uint32_t *)host_target(levels, 4ull * n, &copy_only);
    uint32_t *out = target;
    if (levels && !out && !copy_only) out = whole_stage(g);
    if (!out) out = L.light[0];    // the levels left in flight find no rows
    if (levels)
        hipLaunchKernelGGL(k_wb_out, dim3(grid_for(n, WB_THREADS, 1024)), dim3(WB_THREADS), 0, g->stream, n, level,
                           perm, out);
    GPR_HIP(hipGetLastError());
    GPR_TRY(whole_results(g, out, levels, target));
    info->ms = stream_time_read_ms(g);
    info->iters = (int)h->steps;
    info->push_iters = (int)h->pushes;
    info->edges = h->edges;
    return GPR_OK;
}

int whole_cc(gpr_graph *g, uint32_t *labels, gpr_run_info *info) {
    const uint32_t n = g->n;
    bool copy_only = false;
    uint32_t *const target = (uint32_t *)host_target(labels, 4ull * n, &copy_only);
    uint32_t *out = target;
    if (labels && !out && !copy_only) out = whole_stage(g);
    // the scan scratch holds the parents and, with labels asked for, the
    // recode's minima by original ID (vertices relabelled) or the labels that
    // are copied; both, where there are such labels, want a block
    uint32_t *parent = (uint32_t *)g->scan, *minorig = nullptr;
    WholeMem mem(g);
    if (labels && g->order) minorig = parent + n;
    if (labels && !out) {
        if (minorig) GPR_TRY(mem.take(&out, 4ull * n, "labels"));
        else out = parent + n;
    }
    const unsigned grid = grid_for(n, UF_THREADS, 4096);
    // The run's time ends before the labels go out.  Kernels write the clock
    // (clk) where labels follow: an event between them takes 5 of the 48 us of
    // 4096 vertices.
    volatile unsigned long long *const clk = (unsigned long long *)g->wline;
    unsigned long long *const clk_dev = (unsigned long long *)g->wline_dev;
    if (!labels) stream_time_ms(g, true);
    hipLaunchKernelGGL(k_uf_init, dim3(grid), dim3(UF_THREADS), 0, g->stream, n, g->index, g->nbrs, parent, minorig,
                       clk_dev);
    // a hub next to 1/32 of the vertices, with the smallest ID (relabelled by
    // degree), already holds most of its component: the rounds would cost
    // their launches (10-14 us) and save nothing
    const bool hub = g->order && (uint64_t)g->max_deg * 32 >= n;
    const dim3 fgrid(grid_for(n, LF_THREADS, 1024));
    for (int k = 0; !hub && k < UF_ROUNDS; ++k) {
        if (k == 0)
            hipLaunchKernelGGL(k_uf_flatten, fgrid, dim3(LF_THREADS), 0, g->stream, n, parent, (const uint32_t *)nullptr,
                               (uint32_t *)nullptr);
        hipLaunchKernelGGL(k_uf_round, dim3(grid), dim3(UF_THREADS), 0, g->stream, n, g->index, g->nbrs, parent);
        hipLaunchKernelGGL(k_uf_flatten, fgrid, dim3(LF_THREADS), 0, g->stream, n, parent, (const uint32_t *)nullptr,
                           (uint32_t *)nullptr);
    }
    hipLaunchKernelGGL(k_uf_link, dim3(g->nbuckets + g->nlong_chunks), dim3(UF_THREADS), 0, g->stream, g->nbuckets,
                       g->bucket, g->index, g->nbrs, g->long_rows, g->long_base, g->nlong, parent);
    hipLaunchKernelGGL(k_uf_flatten, fgrid, dim3(LF_THREADS), 0, g->stream, n, parent, g->order, minorig);
    if (labels)
        hipLaunchKernelGGL(k_uf_out, dim3(grid), dim3(UF_THREADS), 0, g->stream, n, parent,
                           g->order ? g->perm : nullptr, minorig, out, clk_dev + 1);
    else
        stream_time_mark(g);
    GPR_HIP(hipGetLastError());
    GPR_TRY(whole_results(g, out, labels, target));
    info->ms = labels ? (double)(clk[1] - clk[0]) / wall_clock_khz() : stream_time_read_ms(g);
    // one step, over every edge
    info->iters = 1;
    info->push_iters = 1;
    info->edges = g->m;
    return GPR_OK;
}

} // namespace gpr
