// label_fold.hpp -- per component, the smallest original ID of its vertices,
// at the component's root (the vertex that carries its own ID as its label).
//
// A giant component sends most vertices to one address: a read before each
// atomic does not help, because every wave in flight reads the unset value
// before the first atomic lands, and those atomics then queue on the address
// (6.1 ms at 33.6M vertices, RMAT; 0.26 ms at 50021).  So a thread keeps one
// label and its minimum in registers, the smaller label of two it meets (a
// label is the smallest internal ID of its component, so a giant's is
// small); the other goes to memory at once.  A wave then folds the lanes that
// hold its smallest label, a workgroup the waves that hold its smallest, and
// one atomic a workgroup is left for a giant: 0.11 ms and 5 us on the same
// graphs.  A root's own ID needs no fold (one vertex a component).
#pragma once
#include "device.hpp"

namespace gpr {

constexpr int LF_THREADS = 256, LF_ITEMS = 8;

__device__ __forceinline__ void label_lower(uint32_t *minorig, uint32_t l, uint32_t o) {
    if (o < __hip_atomic_load(&minorig[l], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&minorig[l], o);
}

struct LabelFold {
    uint32_t l = 0xffffffffu, o = 0xffffffffu;   // the label kept, and its minimum
    // vertex i with label li and original ID oi
    __device__ __forceinline__ void add(uint32_t *minorig, uint64_t i, uint32_t li, uint32_t oi) {
        if (li == i) {
            label_lower(minorig, li, oi);
        } else if (li == l) {
            o = oi < o ? oi : o;
        } else if (li < l) {
            if (l != 0xffffffffu) label_lower(minorig, l, o);
            l = li;
            o = oi;
        } else {
            label_lower(minorig, li, oi);
        }
    }
    // once, by every thread of a workgroup of LF_THREADS
    __device__ __forceinline__ void finish(uint32_t *minorig) {
        __shared__ uint32_t s_l[LF_THREADS / 64], s_o[LF_THREADS / 64];
        const uint32_t wl = wave_min(l);
        const uint32_t wo = wave_min(l == wl ? o : 0xffffffffu);
        if (l != wl && l != 0xffffffffu) label_lower(minorig, l, o);
        if (lane() == 0) {
            s_l[threadIdx.x / 64] = wl;
            s_o[threadIdx.x / 64] = wo;
        }
        __syncthreads();
        if (threadIdx.x != 0) return;
        uint32_t bl = s_l[0], bo = s_o[0];
        for (unsigned j = 1; j < LF_THREADS / 64; ++j) {
            const uint32_t jl = s_l[j], jo = s_o[j];
            if (jl == bl) {
                bo = jo < bo ? jo : bo;
            } else {
                const bool lower = jl < bl;
                const uint32_t fl = lower ? bl : jl, fo = lower ? bo : jo;
                if (fl != 0xffffffffu) label_lower(minorig, fl, fo);
                if (lower) {
                    bl = jl;
                    bo = jo;
                }
            }
        }
        if (bl != 0xffffffffu) label_lower(minorig, bl, bo);
    }
};

} // namespace gpr
