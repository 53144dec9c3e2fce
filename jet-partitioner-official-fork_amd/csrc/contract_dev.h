// Row deduplication steps shared by the contraction kernels. Device only.
#pragma once
#include <hip/hip_runtime.h>

#include "jet_types.h"
#include "wave.h"

namespace jet {

constexpr int32_t EMPTY = -1;

__device__ inline uint32_t slot_hash(vid_t u) { return (uint32_t)u * 0x9E3779B1u; }

// Flattened walk over the edges of a coarse row's fine members mb..me - 1
// (member(x) is the x-th), in chunks of up to 64 members: lane-strided over
// edges, member found by binary search on the chunk's degree prefix held in
// LDS.
template <class M, class F>
__device__ inline void wave_row_edges(const DGraph& g, M&& member, int32_t mb, int32_t me, eoff_t* s_ex, eoff_t* s_rs,
                                      F&& f) {
    const int lane = threadIdx.x & (WAVE - 1);
    for (int32_t m0 = mb; m0 < me; m0 += WAVE) {
        int32_t mi = m0 + lane;
        bool valid = mi < me;
        eoff_t rs = 0, d = 0;
        if (valid) {
            vid_t i = member(mi);
            rs = g.rowptr[i];
            d = g.rowptr[i + 1] - rs;
        }
        eoff_t inc = wave_incl_scan(d);
        eoff_t total = __shfl(inc, WAVE - 1, WAVE);
        s_ex[lane] = inc - d;
        s_rs[lane] = rs;
        int32_t nm = min(WAVE, me - m0);
        wave_sync();
        for (eoff_t fi = lane; fi < total; fi += WAVE) {
            int lo = 0, hi = nm - 1;
            while (lo < hi) {
                int mid = (lo + hi + 1) >> 1;
                if (s_ex[mid] <= fi) lo = mid;
                else hi = mid - 1;
            }
            f(s_rs[lo] + (fi - s_ex[lo]));
        }
        wave_sync();
    }
}

// Adds weight w to key u of an LDS hash table of mask + 1 slots.
__device__ inline void lds_insert(int32_t* keys, int32_t* vals, uint32_t mask, vid_t u, wgt_t w) {
    uint32_t h = slot_hash(u) & mask;
    while (true) {
        int32_t k = keys[h];
        if (k == u) break;
        if (k == EMPTY) {
            int32_t old = atomicCAS(&keys[h], EMPTY, u);
            if (old == EMPTY || old == u) break;
        }
        h = (h + 1) & mask;
    }
    atomicAdd(&vals[h], w);
}

}  // namespace jet
