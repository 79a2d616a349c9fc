// pagerank.hip -- the PageRank edgemap (relax y[d] += contrib[s]) and its
// fused vertex-map tail.
//
// Reference: PRv run loop bench/PRv.C:115-290 (edgemap :202-212, scans and
// maps :214-269), PR_vary run_prec bench/PR_vary.C:247-447 and its encodings
// (customfp.h:20-211, variants :449-648), dense pull over the CSC
// (dsl/emap/GraptorCSCDataParCached.h:60-302 / GraphCSx_csc.h:50-140).
//
// Per iteration, on the handle's stream, with no host round trip (pull; the
// binned sums of pr_cold.hip are the default):
//   k_pr_pull    buckets of <= STREAM_ITEMS rows+edges: neighbour IDs are read
//                coalesced, contributions gathered into LDS, then each row is
//                summed from LDS (lane per short row, wave per row above 64
//                edges).  Rows above LONG_DEG are cut into LONG_CHUNK-edge
//                chunks, one workgroup each, summed by k_pr_long.
//                The last workgroup to finish sums the workgroup partials of
//                y and the maximum of y/deg in a fixed order (FP64) and
//                derives w, 1/s and the FP16 encode scale (pr_fold.hpp);
//                k_pr_reduce does where there are many partials.
//   k_pr_update  x' = (y + w) / s, |x - x'| partials, x = x', contrib =
//                d*x'/deg encoded in the contribution format; the last
//                workgroup sums the residual partials into delta.
// Contributions of every format are accumulated in FP64 registers, as PRv
// does (y_acc is double over FP32 storage, PRv.C:127): a row's sum does not
// depend on whether it is pulled or binned, but for the last rounding.  With
// FP32 registers for 16-bit formats it would (20 iterations on RMAT with 60000
// vertices take 370 us either way, bf16).
#include "internal.hpp"
#include "device.hpp"
#include "pr_codec.hpp"
#include "grid_sync.hpp"
#include "pr_fold.hpp"

#include <math.h>

namespace gpr {

constexpr int PR_THREADS = 256;
constexpr int PR_LDS_EDGES = STREAM_ITEMS + (int)LONG_DEG;
constexpr uint32_t PR_MED = 64;
constexpr int PR_UNROLL = PR_LDS_EDGES / PR_THREADS;  // 16

// PR_UNROLL gathers of one lane, issued back to back: every load is
// unconditional (masked lanes read contrib[0]) and decoding follows all of
// them, so no load waits for the previous one.  Sources at or above
// cold_from (and the 0xffffffff padding) contribute 0.
template <int FMT>
__device__ __forceinline__ void gather_all(const typename Codec<FMT>::store_t *__restrict__ c, const uint32_t *s,
                                           uint32_t cold_from, float *v) {
    typename Codec<FMT>::store_t raw[PR_UNROLL];
#pragma unroll
    for (int u = 0; u < PR_UNROLL; ++u) raw[u] = c[s[u] < cold_from ? s[u] : 0u];
#pragma unroll
    for (int u = 0; u < PR_UNROLL; ++u) v[u] = s[u] < cold_from ? Codec<FMT>::dec(raw[u]) : 0.0f;
}

// Long rows in up to PR_LONG_HERE chunks are folded by the pull's last
// workgroup: a launch less, 5 of an iteration's 20 us on 60000 vertices and
// 1.7M edges.  Above, a thread's chain of chunk loads (8 at a time, 0.7 us
// each) and the rows a thread has would hold the whole chip up, and k_pr_long
// spreads them over workgroups.
constexpr uint32_t PR_LONG_HERE = 256;
template <int FMT>
__global__ void __launch_bounds__(PR_THREADS)
k_pr_pull(uint32_t nbuckets, const uint32_t *__restrict__ bucket, const uint64_t *__restrict__ cindex,
          const uint32_t *__restrict__ cnbrs, const uint32_t *__restrict__ deg,
          const typename Codec<FMT>::store_t *__restrict__ contrib, float *__restrict__ y,
          const uint32_t *__restrict__ long_rows, const uint32_t *__restrict__ long_base, uint32_t nlong,
          double *__restrict__ long_partial, double *part, float *part_max, const PrScalars *prs,
          uint32_t cold_from, PrFold fold, int long_here) {
    __shared__ float vals[PR_LDS_EDGES];
    __shared__ uint32_t rs[STREAM_ITEMS + 1];
    __shared__ uint32_t medq[PR_LDS_EDGES / PR_MED + 1];
    __shared__ uint32_t nmed;
    __shared__ double dred[PR_THREADS / 64];
    __shared__ float fred[PR_THREADS / 64];
    __shared__ int s_last;
    const float dscale = FMT == GPR_CONTRIB_F16 ? 1.0f / prs->enc_scale : 1.0f;
    const uint32_t b = blockIdx.x;
    if (b >= nbuckets) {
        // ---- one chunk of a long row
        const uint32_t c = b - nbuckets;
        uint32_t lo = 0, hi = nlong;
        while (lo < hi) {
            uint32_t mid = (lo + hi) >> 1;
            if (long_base[mid] <= c) lo = mid + 1; else hi = mid;
        }
        const uint32_t li = lo - 1;
        const uint32_t row = long_rows[li];
        const uint64_t rb = cindex[row], re = cindex[row + 1];
        const uint64_t cb = rb + (uint64_t)(c - long_base[li]) * LONG_CHUNK;
        const uint64_t ce = min(re, cb + LONG_CHUNK);
        double acc = 0.0;
        // PR_UNROLL independent neighbour loads, then as many gathers, in
        // flight per lane
        for (uint64_t base = cb; base < ce; base += (uint64_t)PR_THREADS * PR_UNROLL) {
            uint32_t s[PR_UNROLL];
#pragma unroll
            for (int u = 0; u < PR_UNROLL; ++u) {
                const uint64_t e = base + (uint64_t)u * PR_THREADS + threadIdx.x;
                s[u] = e < ce ? cnbrs[e] : 0xffffffffu;
            }
            float v[PR_UNROLL];
            gather_all<FMT>(contrib, s, cold_from, v);
#pragma unroll
            for (int u = 0; u < PR_UNROLL; ++u) acc += (double)v[u];
        }
        double tot = block_sum(acc, dred);
        if (threadIdx.x == 0) {
            st_part(&long_partial[c], tot);
            st_part(&part[b], 0.0);
            st_part(&part_max[b], 0.0f);
        }
        if (!long_here) return;   // the fold is k_pr_long's
    } else {
        // ---- a bucket of rows
        const uint32_t r0 = bucket[b], r1 = bucket[b + 1];
        double my_sum = 0.0;
        float my_max = 0.0f;
        if (r0 < r1) {
            uint32_t r1x = r1;
            if (cindex[r1] - cindex[r1 - 1] > LONG_DEG) r1x = r1 - 1;
            const uint64_t e0 = cindex[r0];
            const uint32_t nrows = r1x - r0;
            const uint32_t ne = (uint32_t)(cindex[r1x] - e0);
            if (threadIdx.x == 0) nmed = 0;
            for (uint32_t base = 0; base <= nrows; base += PR_THREADS * 8) {
                uint64_t ix[8];
    #pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint32_t i = base + u * PR_THREADS + threadIdx.x;
                    ix[u] = i <= nrows ? cindex[r0 + i] : 0;
                }
    #pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint32_t i = base + u * PR_THREADS + threadIdx.x;
                    if (i <= nrows) rs[i] = (uint32_t)(ix[u] - e0);
                }
            }
            // (plain loads: a small graph's neighbours stay in the L2s from one
            // iteration to the next; non-temporal ones took 46 us instead of 39
            // an iteration on 7.6M edges)
            // a bucket holds < PR_LDS_EDGES edges: one round of PR_UNROLL
            // independent neighbour loads and gathers per lane covers it
            for (uint32_t base = 0; base < ne; base += PR_THREADS * PR_UNROLL) {
                uint32_t s[PR_UNROLL];
    #pragma unroll
                for (int u = 0; u < PR_UNROLL; ++u) {
                    const uint32_t i = base + u * PR_THREADS + threadIdx.x;
                    s[u] = i < ne ? cnbrs[e0 + i] : 0xffffffffu;
                }
                float v[PR_UNROLL];
                gather_all<FMT>(contrib, s, cold_from, v);
    #pragma unroll
                for (int u = 0; u < PR_UNROLL; ++u) {
                    const uint32_t i = base + u * PR_THREADS + threadIdx.x;
                    if (i < ne) vals[i] = v[u];
                }
            }
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < nrows; i += PR_THREADS) {
                const uint32_t a = rs[i], z = rs[i + 1];
                if (z - a > PR_MED) {
                    medq[atomicAdd(&nmed, 1u)] = i;
                    continue;
                }
                double acc = 0.0;
                for (uint32_t j = a; j < z; ++j) acc += (double)vals[j];
                const float yv = (float)acc * dscale;
                y[r0 + i] = yv;
                my_sum += (double)yv;
                if (FMT == GPR_CONTRIB_F16) {
                    const uint32_t dg = deg[r0 + i];
                    if (dg) my_max = fmaxf(my_max, yv / (float)dg);
                }
            }
            __syncthreads();
            const uint32_t nm = nmed;
            const unsigned w = threadIdx.x / 64, ln = lane();
            for (uint32_t q = w; q < nm; q += PR_THREADS / 64) {
                const uint32_t i = medq[q];
                const uint32_t a = rs[i], z = rs[i + 1];
                double acc = 0.0;
                for (uint32_t j = a + ln; j < z; j += 64) acc += (double)vals[j];
                acc = wave_sum(acc);
                if (ln == 0) {
                    const float yv = (float)acc * dscale;
                    y[r0 + i] = yv;
                    my_sum += (double)yv;
                    if (FMT == GPR_CONTRIB_F16) {
                        const uint32_t dg = deg[r0 + i];
                        if (dg) my_max = fmaxf(my_max, yv / (float)dg);
                    }
                }
            }
        }
        const double ts = block_sum(my_sum, dred);
        my_max = wave_max(my_max);
        __syncthreads();
        if (lane() == 0) fred[threadIdx.x / 64] = my_max;
        __syncthreads();
        if (threadIdx.x == 0) {
            float mx = fred[0];
            for (int i = 1; i < PR_THREADS / 64; ++i) mx = fmaxf(mx, fred[i]);
            st_part(&part[b], ts);
            st_part(&part_max[b], mx);
        }
    }
    constexpr bool F16 = FMT == GPR_CONTRIB_F16;
    if (!long_here) {
        pr_fold_sum<PR_THREADS, F16>(fold, part, part_max, dred, &s_last);
        return;
    }
    // the last workgroup folds the long rows too (k_pr_long)
    if (!last_workgroup(fold.ticket, &s_last)) return;
    double s = part_sum<PR_THREADS, 1>(part, gridDim.x);
    float m = F16 ? part_max_of<PR_THREADS>(part_max, gridDim.x) : 0.0f;
    for (uint32_t li = threadIdx.x; li < nlong; li += PR_THREADS) {
        const uint32_t c1 = long_base[li + 1], row = long_rows[li];
        double t = 0.0;
        for (uint32_t c = long_base[li]; c < c1; c += PART_U) {
            double v[PART_U];
#pragma unroll
            for (int u = 0; u < PART_U; ++u) v[u] = ld_part(&long_partial[c + u < c1 ? c + u : c]);
#pragma unroll
            for (int u = 0; u < PART_U; ++u)
                if (c + u < c1) t += v[u];
        }
        const float yv = (float)t * dscale;
        y[row] = yv;
        s += (double)yv;
        if (F16) {
            const uint32_t dg = deg[row];
            if (dg) m = fmaxf(m, yv / (float)dg);
        }
    }
    pr_fold_shares<PR_THREADS, F16>(fold, s, m, dred);
}

// One thread per long row: fold its chunk partials in chunk order.
template <bool F16>
__global__ void __launch_bounds__(PR_THREADS)
k_pr_long(uint32_t nlong, const uint32_t *__restrict__ long_rows, const uint32_t *__restrict__ long_base,
          const double *__restrict__ long_partial, const uint32_t *__restrict__ deg, float *y,
          double *part, float *part_max, uint32_t slot0, const PrScalars *prs, PrFold fold) {
    __shared__ double dred[PR_THREADS / 64];
    __shared__ int s_last;
    const float dscale = F16 ? 1.0f / prs->enc_scale : 1.0f;
    for (uint32_t li = blockIdx.x * blockDim.x + threadIdx.x; li < nlong; li += gridDim.x * blockDim.x) {
        double s = 0.0;
        for (uint32_t c = long_base[li]; c < long_base[li + 1]; ++c) s += long_partial[c];
        const uint32_t row = long_rows[li];
        const float yv = (float)s * dscale;
        y[row] = yv;
        st_part(&part[slot0 + li], (double)yv);
        const uint32_t dg = deg[row];
        st_part(&part_max[slot0 + li], dg ? yv / (float)dg : 0.0f);
    }
    // every thread wrote partials: all of the workgroup's are acknowledged
    // before its thread 0 counts it
    __builtin_amdgcn_s_waitcnt(WAIT_VM0);
    __syncthreads();
    pr_fold_sum<PR_THREADS, F16>(fold, part, part_max, dred, &s_last);
}

// Deterministic reduction of `count` partial sums and maxima by many
// workgroups, for pulls of more than PR_FOLD_MAX partials: the last
// workgroup sets the scalars (set_sum) or leaves the slices' maxima to
// k_pr_set_scale.
constexpr int RED_THREADS = 256;
constexpr int RED_BLOCKS = 64;
// partials a pull's own last workgroup folds (64 loads a thread)
constexpr uint32_t PR_FOLD_MAX = 16384;
__global__ void __launch_bounds__(RED_THREADS)
k_pr_reduce(const double *__restrict__ part, const float *__restrict__ part_max, uint32_t count, double *slices,
            unsigned int *ticket, PrScalars *prs, int set_sum, uint32_t n, float damping, int f16) {
    __shared__ double r1[RED_THREADS];
    __shared__ float r3[RED_THREADS];
    __shared__ int s_last;
    const uint32_t per = (count + gridDim.x - 1) / gridDim.x;
    const uint32_t lo = blockIdx.x * per, hi = min(count, lo + per);
    double s1 = 0.0;
    float mx = 0.0f;
    for (uint32_t i = lo + threadIdx.x; i < hi; i += RED_THREADS) {
        s1 += part[i];
        mx = fmaxf(mx, part_max[i]);
    }
    r1[threadIdx.x] = s1;
    r3[threadIdx.x] = mx;
    __syncthreads();
    for (int o = RED_THREADS / 2; o > 0; o >>= 1) {
        if (threadIdx.x < (unsigned)o) {
            r1[threadIdx.x] += r1[threadIdx.x + o];
            r3[threadIdx.x] = fmaxf(r3[threadIdx.x], r3[threadIdx.x + o]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        st_part(&slices[2 * blockIdx.x], r1[0]);
        st_part(&slices[2 * blockIdx.x + 1], (double)r3[0]);
    }
    if (!last_workgroup(ticket, &s_last) || threadIdx.x != 0 || !set_sum) return;
    double a = 0.0, m = 0.0;
    for (unsigned i = 0; i < gridDim.x; ++i) {
        a += ld_part(&slices[2 * i]);
        m = fmax(m, ld_part(&slices[2 * i + 1]));
    }
    if (f16) pr_set_sum<true>(prs, a, m, n, damping);
    else pr_set_sum<false>(prs, a, m, n, damping);
}

// Bound by its streams (20 B a vertex in FP32).  The last workgroup also
// sums the residual and the ranks, into the device's scalars and the host's
// line.
//
// FUSED (gpr_pr_iterate_fused where the edgemap pulls): no residual, and x
// unwritten when null.
constexpr int PR_UPDATE_U = 4;
template <int FMT, bool FUSED>
__global__ void __launch_bounds__(256)
k_pr_update(uint32_t n, const float *__restrict__ y, float *__restrict__ x, typename Codec<FMT>::store_t *contrib,
            const uint32_t *__restrict__ deg, float damping, PrScalars *prs, double *part_delta, double *part_sums,
            unsigned int *ticket, HostScalars *h) {
    __shared__ double r1[4], r2[4];
    __shared__ int s_last;
    const double w = prs->w, inv_s = prs->inv_s;
    const float sc = FMT == GPR_CONTRIB_F16 ? prs->enc_scale : 1.0f;
    double dl = 0.0, sx = 0.0;
    const uint64_t step = (uint64_t)gridDim.x * 256;
    for (uint64_t v0 = blockIdx.x * 256 + threadIdx.x; v0 < n; v0 += step * PR_UPDATE_U) {
        float yv[PR_UPDATE_U], xv[PR_UPDATE_U];
        uint32_t dg[PR_UPDATE_U];
#pragma unroll
        for (int u = 0; u < PR_UPDATE_U; ++u) {
            const uint64_t v = v0 + u * step < n ? v0 + u * step : v0;
            yv[u] = y[v];
            if constexpr (!FUSED) xv[u] = x[v];
            dg[u] = deg[v];
        }
#pragma unroll
        for (int u = 0; u < PR_UPDATE_U; ++u) {
            const uint64_t v = v0 + u * step;
            if (v >= n) break;
            const float xn = (float)(((double)yv[u] + w) * inv_s);
            if constexpr (!FUSED) {
                dl += (double)fabsf(xv[u] - xn);
                sx += (double)xn;
            }
            if (!FUSED || x) x[v] = xn;
            const float cv = dg[u] ? damping * xn / (float)dg[u] : 0.0f;
            contrib[v] = Codec<FMT>::enc(cv * sc);
        }
    }
    if constexpr (FUSED) return;
    dl = block_sum(dl, r1);
    sx = block_sum(sx, r2);
    if (threadIdx.x == 0) {
        st_part(&part_delta[blockIdx.x], dl);
        st_part(&part_sums[blockIdx.x], sx);
    }
    if (!last_workgroup(ticket, &s_last)) return;
    dl = block_sum(part_sum<256, 1>(part_delta, gridDim.x), r1);
    sx = block_sum(part_sum<256, 1>(part_sums, gridDim.x), r2);
    if (threadIdx.x == 0) {
        prs->delta = dl;
        prs->sum_x = sx;
        h->delta = dl;
        h->sum_x = sx;
    }
}

// contrib = d*x/deg from the current ranks (start of a run or of a stage).
template <int FMT>
__global__ void __launch_bounds__(256)
k_pr_contrib(uint32_t n, const float *__restrict__ x, typename Codec<FMT>::store_t *contrib,
             const uint32_t *__restrict__ deg, float damping, const PrScalars *__restrict__ prs) {
    const float sc = FMT == GPR_CONTRIB_F16 ? prs->enc_scale : 1.0f;
    for (uint32_t v = blockIdx.x * 256 + threadIdx.x; v < n; v += gridDim.x * 256) {
        const uint32_t dg = deg[v];
        const float cv = dg ? damping * x[v] / (float)dg : 0.0f;
        contrib[v] = Codec<FMT>::enc(cv * sc);
    }
}

__global__ void __launch_bounds__(256)
k_pr_xmax(uint32_t n, const float *__restrict__ x, double *part, float *part_max) {
    __shared__ float fr[4];
    float mx = 0.0f;
    for (uint32_t v = blockIdx.x * 256 + threadIdx.x; v < n; v += gridDim.x * 256) mx = fmaxf(mx, x[v]);
    mx = wave_max(mx);
    if (lane() == 0) fr[threadIdx.x / 64] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        part[blockIdx.x] = 0.0;
        part_max[blockIdx.x] = fmaxf(fmaxf(fr[0], fr[1]), fmaxf(fr[2], fr[3]));
    }
}

__global__ void k_pr_set_scale(PrScalars *prs, const double *slices, uint32_t nslices, float damping, int f16) {
    if (threadIdx.x != 0) return;
    double m = 0.0;
    for (uint32_t i = 0; i < nslices; ++i) m = fmax(m, slices[2 * i + 1]);
    if (f16) {
        const double u = (double)damping * m;
        int k = u > 0.0 ? (int)floor(log2(32768.0 / u)) : 0;
        k = k > 100 ? 100 : k < -100 ? -100 : k;
        prs->enc_scale = (float)ldexp(1.0, k);
    } else {
        prs->enc_scale = 1.0f;
    }
}

// ---- host side -----------------------------------------------------------------
static size_t fmt_bytes(int fmt) { return fmt == GPR_CONTRIB_F32 ? 4 : 2; }

static unsigned update_grid(uint32_t n) { return grid_for(n, 256, 2048); }

// First cold source of the PageRank edgemap: sources at or above it are
// summed through the binned layout (pr_cold.hip), those below by the pull.
// The split is the FP32 bytes of pulled contributions (tunable
// pr_split_bytes): 0 bins every edge, >= 4n pulls every edge.
static uint32_t split_point(gpr_graph *g) {
    const double h = floor(tun().pr_split_bytes / 4.0);
    return h >= (double)g->n ? g->n : (uint32_t)h;
}

// Whether the automatic split (pr_split_bytes 0) pulls every edge instead of
// binning it.  Binned sums take up to four launches an iteration,
// with every bin cleared and written out, and pay it back by streaming; a pull is two launches, and its
// gathers run at 200 G/s and more while the contributions stay in an XCD's
// 4 MB L2.  PRv per iteration, pull against bins (FP32): RMAT with 0.1M
// edges 12 / 25 us, 1.8M 19 / 35, 7.6M 39 / 53, 15M 73 / 71, 31M 129 / 91;
// uniform random with 8M edges on 1M vertices 64 / 70.  So up to
// pr_pull_edges (2^23) edges, on at most 2^20 vertices.  A new graph is
// spared the layout's construction as well.
static bool pulls_all(const gpr_graph *g) {
    return tun().pr_split_bytes < 4.0 && (double)g->m <= tun().pr_pull_edges && g->n <= (1u << 20);
}

// x_tail != nullptr: the previous iteration's tail is fused into the write
// stage (the caller has checked cold_tail_fusable after cold_prepare)
static int pr_edgemap_impl(gpr_graph *g, const gpr_emap_desc *desc, gpr_frontier *in, gpr_iter_stats *st,
                           float *x_tail) {
    GPR_REQUIRE(!in || in->kind == GPR_FRONTIER_ALL, "PR edgemap runs over the all-true frontier only");
    GPR_REQUIRE(desc->prop && desc->prop->dtype == GPR_F32, "PR edgemap: accumulator must be an f32 property");
    const int fmt = desc->contrib_fmt;
    GPR_REQUIRE(fmt >= GPR_CONTRIB_F32 && fmt <= GPR_CONTRIB_SCFP16, "PR edgemap: unknown contribution format %d", fmt);
    GPR_REQUIRE(desc->contrib && desc->contrib->elem == fmt_bytes(fmt),
                "PR edgemap: contribution property has the wrong element size for format %d", fmt);
    uint32_t cold_from = pulls_all(g) ? g->n : split_point(g);
    if (cold_from < g->n) {
        GPR_TRY(cold_prepare(g, cold_from));
        if (g->cold->ntiles == 0) cold_from = g->n;   // no cold edges
    }
    const bool split = cold_from < g->n;
    const uint32_t nblk = g->nbuckets + g->nlong_chunks;
    size_t need = (size_t)nblk + g->nlong + 4096;
    if (split) need += g->cold->nbins + (size_t)g->cold->nmulti * (COLD_BIN / 1024);
    GPR_TRY(ensure_partials(g, need));
    float *y = (float *)desc->prop->d;
    const void *cb = desc->contrib->d;
    const float damping = desc->damping > 0.f ? desc->damping : 0.85f;
    if (st) GPR_HIP(hipEventRecord(g->ev0, g->stream));
    if (split) {
        ProfScope ps(g, "pr_cold_write");
        GPR_TRY(cold_launch_write(g, fmt, cb, y, x_tail, damping));
    }
    // the kernel that writes the last of y's partials also folds them into
    // the scalars: the binned sums' last kernel; without them the pull, or
    // the long rows' kernel after it
    const uint32_t nparts = nblk + g->nlong;
    PrFold fold = {g->ticket, g->prs, split || nparts > PR_FOLD_MAX ? 0 : nparts, g->n, damping};
    PrFold pull_fold = fold;
    const int long_here = fold.count && g->nlong && g->nlong_chunks <= PR_LONG_HERE;
    if (g->nlong && !long_here) pull_fold.count = 0;
    if (cold_from > 0) {
        // the pull over sources [0, cold_from); every source when not split
        ProfScope ps(g, "pr_pull");
#define PR_PULL(F)                                                                                              \
    hipLaunchKernelGGL(k_pr_pull<F>, dim3(nblk), dim3(PR_THREADS), 0, g->stream, g->nbuckets, g->bucket,        \
                       g->cindex, g->cnbrs, g->deg, (const typename Codec<F>::store_t *)cb, y, g->long_rows,   \
                       g->long_base, g->nlong, g->long_partial, g->partial, g->partial_f, g->prs, cold_from, pull_fold,    \
                       long_here)
        switch (fmt) {
        case GPR_CONTRIB_F32: PR_PULL(GPR_CONTRIB_F32); break;
        case GPR_CONTRIB_BF16: PR_PULL(GPR_CONTRIB_BF16); break;
        case GPR_CONTRIB_F16: PR_PULL(GPR_CONTRIB_F16); break;
        case GPR_CONTRIB_CFP16: PR_PULL(GPR_CONTRIB_CFP16); break;
        case GPR_CONTRIB_BF16T: PR_PULL(GPR_CONTRIB_BF16T); break;
        case GPR_CONTRIB_SCFP16: PR_PULL(GPR_CONTRIB_SCFP16); break;
        }
#undef PR_PULL
    }
    if (cold_from > 0 && g->nlong && !long_here) {
        ProfScope ps(g, "pr_long");
#define PR_LONG(F16)                                                                                            \
    hipLaunchKernelGGL(k_pr_long<F16>, dim3(grid_for(g->nlong, PR_THREADS, 1024)), dim3(PR_THREADS), 0, g->stream, \
                       g->nlong, g->long_rows, g->long_base, g->long_partial, g->deg, y, g->partial, g->partial_f, \
                       nblk, g->prs, fold)
        if (fmt == GPR_CONTRIB_F16) PR_LONG(true); else PR_LONG(false);
#undef PR_LONG
    }
    if (split) {
        // y (+)= the binned sums; their per-bin partials replace the pull's
        ProfScope ps(g, "pr_cold_accum");
        GPR_TRY(cold_launch_accum(g, fmt, y, cold_from > 0 ? 1 : 0, g->partial, g->partial_f, damping));
    } else if (!fold.count) {
        ProfScope ps(g, "pr_reduce");
        hipLaunchKernelGGL(k_pr_reduce, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, g->stream, g->partial, g->partial_f,
                           nparts, g->dsum_slices, g->ticket, g->prs, 1, g->n, damping,
                           fmt == GPR_CONTRIB_F16);
    }
    GPR_HIP(hipGetLastError());
    if (st) {
        GPR_HIP(hipEventRecord(g->ev1, g->stream));
        gpr_iter_stats s = {};
        s.nactv_in = g->n;
        s.nacte_in = g->m;
        s.direction = GPR_DIR_PULL;
        s.edges_scanned = g->m;
        GPR_HIP(hipEventSynchronize(g->ev1));
        float ms = 0.f;
        GPR_HIP(hipEventElapsedTime(&ms, g->ev0, g->ev1));
        s.ms = ms;
        *st = s;
    }
    return GPR_OK;
}

// x' and its contributions from y; the residual too unless fused.
static int launch_update(gpr_graph *g, int fmt, bool fused, const float *y, float *x, void *contrib, float damping) {
    const uint32_t n = g->n;
    const unsigned grid = update_grid(n);
    GPR_TRY(ensure_partials(g, 2 * (size_t)grid + 64));
    ProfScope ps(g, "pr_update");
#define PR_UPDATE_(F, U)                                                                                       \
    hipLaunchKernelGGL((k_pr_update<F, U>), dim3(grid), dim3(256), 0, g->stream, n, y, x,                       \
                       (typename Codec<F>::store_t *)contrib, g->deg, damping, g->prs, g->partial,             \
                       g->partial + grid, g->ticket, g->hsc_dev)
#define PR_UPDATE(F)                                                                                           \
    if (fused) PR_UPDATE_(F, true); else PR_UPDATE_(F, false)
    switch (fmt) {
    case GPR_CONTRIB_F32: PR_UPDATE(GPR_CONTRIB_F32); break;
    case GPR_CONTRIB_BF16: PR_UPDATE(GPR_CONTRIB_BF16); break;
    case GPR_CONTRIB_F16: PR_UPDATE(GPR_CONTRIB_F16); break;
    case GPR_CONTRIB_CFP16: PR_UPDATE(GPR_CONTRIB_CFP16); break;
    case GPR_CONTRIB_BF16T: PR_UPDATE(GPR_CONTRIB_BF16T); break;
    case GPR_CONTRIB_SCFP16: PR_UPDATE(GPR_CONTRIB_SCFP16); break;
    }
#undef PR_UPDATE
#undef PR_UPDATE_
    GPR_HIP(hipGetLastError());
    return GPR_OK;
}

int pr_edgemap(gpr_graph *g, const gpr_emap_desc *desc, gpr_frontier *in, gpr_iter_stats *st) {
    return pr_edgemap_impl(g, desc, in, st, nullptr);
}

} // namespace gpr

using namespace gpr;

extern "C" int gpr_pr_iterate_fused(gpr_graph *g, gpr_prop *x, gpr_prop *y, int fmt, float damping, int flags,
                                    gpr_iter_stats *st) {
    if (!g || !x || !y || x->dtype != GPR_F32 || y->dtype != GPR_F32 || x->g != g || y->g != g) return GPR_E_INVAL;
    GPR_REQUIRE(fmt >= GPR_CONTRIB_F32 && fmt <= GPR_CONTRIB_SCFP16, "pr_iterate_fused: unknown format %d", fmt);
    GPR_REQUIRE(split_point(g) == 0, "pr_iterate_fused: needs every edge binned (pr_split_bytes 0)");
    const bool pull = pulls_all(g);
    if (!pull) GPR_TRY(cold_prepare(g, 0));
    GPR_REQUIRE(pull ? g->m > 0 : cold_tail_fusable(g), "pr_iterate_fused: the graph has no binned edges");
    gpr_emap_desc d = {};
    d.relax = GPR_RELAX_PR_SUM;
    d.prop = y;
    d.contrib_fmt = fmt;
    d.damping = damping;
    // the contribution property is never read by the write stage, which
    // computes the contributions: a stand-in of the right element size
    // passes the checks.  A pull reads them from the handle's scratch.
    gpr_prop stand_in = *y;
    stand_in.elem = (uint32_t)fmt_bytes(fmt);
    d.contrib = &stand_in;
    if (pull) {
        if (!g->pr_contrib)
            GPR_TRY(dev_alloc((void **)&g->pr_contrib, sizeof(float) * (size_t)g->n, "pagerank contributions"));
        stand_in.d = g->pr_contrib;
        GPR_TRY(launch_update(g, fmt, true, (const float *)y->d, flags & GPR_PR_SKIP_RANKS ? nullptr : (float *)x->d,
                              g->pr_contrib, damping > 0.f ? damping : 0.85f));
        return pr_edgemap_impl(g, &d, nullptr, st, nullptr);
    }
    g->pr_skip_unlinked = (flags & (GPR_PR_SKIP_UNLINKED | GPR_PR_SKIP_RANKS)) != 0;
    g->pr_skip_ranks = (flags & GPR_PR_SKIP_RANKS) != 0;
    const int r = pr_edgemap_impl(g, &d, nullptr, st, (float *)x->d);
    g->pr_skip_unlinked = false;
    g->pr_skip_ranks = false;
    return r;
}

extern "C" int gpr_pr_contrib(gpr_graph *g, const gpr_prop *x, gpr_prop *contrib, int fmt, float damping) {
    if (!g || !x || !contrib || x->dtype != GPR_F32) return GPR_E_INVAL;
    GPR_REQUIRE(fmt >= GPR_CONTRIB_F32 && fmt <= GPR_CONTRIB_SCFP16 && contrib->elem == fmt_bytes(fmt),
                "pr_contrib: bad contribution format %d / property", fmt);
    const uint32_t n = g->n;
    const unsigned grid = update_grid(n);
    GPR_TRY(ensure_partials(g, grid + 64));
    if (fmt == GPR_CONTRIB_F16) {
        hipLaunchKernelGGL(k_pr_xmax, dim3(grid), dim3(256), 0, g->stream, n, (const float *)x->d, g->partial,
                           g->partial_f);
        hipLaunchKernelGGL(k_pr_reduce, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, g->stream, g->partial, g->partial_f,
                           grid, g->dsum_slices, g->ticket, g->prs, 0, n, damping, 0);
        hipLaunchKernelGGL(k_pr_set_scale, dim3(1), dim3(64), 0, g->stream, g->prs, g->dsum_slices, RED_BLOCKS,
                           damping, 1);
    } else {
        hipLaunchKernelGGL(k_pr_set_scale, dim3(1), dim3(64), 0, g->stream, g->prs, g->dsum_slices, 0, damping, 0);
    }
#define PR_CONTRIB(F)                                                                                          \
    hipLaunchKernelGGL(k_pr_contrib<F>, dim3(grid), dim3(256), 0, g->stream, n, (const float *)x->d,            \
                       (typename Codec<F>::store_t *)contrib->d, g->deg, damping, g->prs)
    switch (fmt) {
    case GPR_CONTRIB_F32: PR_CONTRIB(GPR_CONTRIB_F32); break;
    case GPR_CONTRIB_BF16: PR_CONTRIB(GPR_CONTRIB_BF16); break;
    case GPR_CONTRIB_F16: PR_CONTRIB(GPR_CONTRIB_F16); break;
    case GPR_CONTRIB_CFP16: PR_CONTRIB(GPR_CONTRIB_CFP16); break;
    case GPR_CONTRIB_BF16T: PR_CONTRIB(GPR_CONTRIB_BF16T); break;
    case GPR_CONTRIB_SCFP16: PR_CONTRIB(GPR_CONTRIB_SCFP16); break;
    }
#undef PR_CONTRIB
    GPR_HIP(hipGetLastError());
    return GPR_OK;
}

extern "C" int gpr_pr_finish(gpr_graph *g, gpr_prop *x, const gpr_prop *y, gpr_prop *contrib, int fmt, float damping,
                             double *delta, double *sum_x) {
    if (!g || !x || !y || !contrib || x->dtype != GPR_F32 || y->dtype != GPR_F32) return GPR_E_INVAL;
    GPR_REQUIRE(fmt >= GPR_CONTRIB_F32 && fmt <= GPR_CONTRIB_SCFP16 && contrib->elem == fmt_bytes(fmt),
                "pr_finish: bad contribution format %d / property", fmt);
    GPR_TRY(launch_update(g, fmt, false, (const float *)y->d, (float *)x->d, contrib->d, damping));
    if (delta || sum_x) {
        GPR_HIP(hipStreamSynchronize(g->stream));
        if (delta) *delta = g->hsc->delta;
        if (sum_x) *sum_x = g->hsc->sum_x;
    }
    return GPR_OK;
}

extern "C" int gpr_pr_scalars(gpr_graph *g, double *sum_y, double *delta, double *sum_x, float *enc_scale) {
    if (!g) return GPR_E_INVAL;
    if (!sum_y && !enc_scale) {
        GPR_HIP(hipStreamSynchronize(g->stream));
        if (delta) *delta = g->hsc->delta;
        if (sum_x) *sum_x = g->hsc->sum_x;
        return GPR_OK;
    }
    PrScalars h;
    GPR_HIP(hipMemcpyAsync(&h, g->prs, sizeof(h), hipMemcpyDeviceToHost, g->stream));
    GPR_HIP(hipStreamSynchronize(g->stream));
    if (sum_y) *sum_y = h.sum_y;
    if (delta) *delta = h.delta;
    if (sum_x) *sum_x = h.sum_x;
    if (enc_scale) *enc_scale = h.enc_scale;
    return GPR_OK;
}
