// pr_fold.hpp -- the scalars of a PageRank iteration from its partial sums,
// computed by the last workgroup of the kernel that writes the partials.
#pragma once
#include "device.hpp"
#include "grid_sync.hpp"

namespace gpr {

// What the last workgroup folds: count partials (and maxima), by its
// threads in a fixed order, so that the sums do not depend on which
// workgroup comes last.
struct PrFold {
    unsigned int *ticket;
    PrScalars *prs;
    uint32_t count;      // partials; 0: no fold in this kernel
    uint32_t n;
    float damping;
};

// Sum of y known: PRv.C:214-240, w = (1 - s)/n; y += w; s = sum y; y *= 1/s.
// sum(y + w) = s + n*w is formed analytically in FP64.  FP16: the encode
// scale from m, the largest y/deg.
template <bool F16>
__device__ __forceinline__ void pr_set_sum(PrScalars *prs, double a, double m, uint32_t n, float damping) {
    const double w = (1.0 - a) / (double)n;
    const double s2t = a + (double)n * w;
    prs->sum_y = a;
    prs->w = w;
    prs->inv_s = 1.0 / s2t;
    prs->max_ratio = (float)m;
    if constexpr (F16) {
        // largest next contribution <= d * (max y/deg + w) / s; keep it
        // at or below 2^15 so the FP16 store cannot overflow (max 65504)
        const double u = (double)damping * (m + w) / s2t;
        int k = u > 0.0 ? (int)floor(log2(32768.0 / u)) : 0;
        k = k > 100 ? 100 : k < -100 ? -100 : k;
        prs->enc_scale = (float)ldexp(1.0, k);
    } else {
        prs->enc_scale = 1.0f;
    }
}

// The scalars from this thread's shares s and m of the sum and the maximum, by
// all threads of the last workgroup.
template <int NT, bool F16>
__device__ __forceinline__ void pr_fold_shares(const PrFold &f, double s, float m, double *dred) {
    const double a = block_sum(s, dred);
    double mx = 0.0;
    if constexpr (F16) {
        m = wave_max(m);
        __syncthreads();
        if (lane() == 0) dred[threadIdx.x / 64] = (double)m;
        __syncthreads();
        for (int i = 0; i < NT / 64; ++i) mx = fmax(mx, dred[i]);
    }
    if (threadIdx.x == 0) pr_set_sum<F16>(f.prs, a, mx, f.n, f.damping);
}
template <int NT>
__device__ __forceinline__ float part_max_of(const float *part_max, uint32_t count) {
    float m = 0.0f;
    for (uint32_t i = threadIdx.x; i < count; i += NT) m = fmaxf(m, ld_part(&part_max[i]));
    return m;
}

// The end of a kernel whose workgroups wrote part[] and part_max[] (thread
// 0, st_part): the last one sets the scalars.  dred: NT/64 doubles of LDS.
template <int NT, bool F16>
__device__ __forceinline__ void pr_fold_sum(const PrFold &f, const double *part, const float *part_max, double *dred,
                                            int *s_last) {
    if (!f.count || !last_workgroup(f.ticket, s_last)) return;
    pr_fold_shares<NT, F16>(f, part_sum<NT, 1>(part, f.count), F16 ? part_max_of<NT>(part_max, f.count) : 0.0f, dred);
}

} // namespace gpr
