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

// The edges ea..eb - 1 of the coarse rows' concatenated fine edges, all of one
// row with members mb..me - 1, by a wave: moff[x] is the first edge of the x-th
// member. f(j, e) gets the fine edge's index and its place. s_e, s_rs: WAVE
// entries of the wave's own.
template <class F>
__device__ inline void wave_edge_range(const DGraph& g, const vid_t* members, const eoff_t* moff, int32_t mb,
                                       int32_t me, eoff_t ea, eoff_t eb, int32_t* s_e, eoff_t* s_rs, F&& f) {
    const int lane = threadIdx.x & (WAVE - 1);
    int32_t lo = mb, hi = me - 1;  // the member that holds edge ea
    while (lo < hi) {
        const int32_t mid = lo + (hi - lo + 1) / 2;
        if (moff[mid] <= ea) lo = mid;
        else hi = mid - 1;
    }
    for (int32_t m0 = lo; ea < eb && m0 < me; m0 += WAVE) {
        // offsets within the range: a member that began before it starts at 0
        const bool in = m0 + lane < me;
        eoff_t rel = in ? moff[m0 + lane] - ea : INT32_MAX;
        eoff_t rs = in ? g.rowptr[members[m0 + lane]] : 0;
        if (rel < 0) {
            rs -= rel;
            rel = 0;
        }
        s_e[lane] = rel < INT32_MAX ? (int32_t)rel : INT32_MAX;
        s_rs[lane] = rs;
        wave_sync();
        const eoff_t wend = m0 + WAVE < me ? min(eb, moff[m0 + WAVE]) : eb;
        for (int32_t x = lane; x < (int32_t)(wend - ea); x += WAVE) {
            int q = 0;  // the last member that starts at or before x
            for (int step = WAVE / 2; step >= 1; step >>= 1)
                if (s_e[q + step] <= x) q += step;
            f(s_rs[q] + (x - s_e[q]), ea + x);
        }
        wave_sync();
        if (wend > ea) ea = wend;
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
