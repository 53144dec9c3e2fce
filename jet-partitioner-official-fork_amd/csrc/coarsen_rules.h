// Choices shared by the coarsening kernels (src/heuristics.hpp). Device only.
#pragma once
#include "jet_types.h"

namespace jet {

// pickMatch choice: lexicographic max of (weight, xorshift32(v + r)) over
// eligible neighbours with weight >= 0 (weight ignored when uniform).
__device__ inline void pick_better(int64_t& bw, uint32_t& bh, vid_t& bv, int64_t w, uint32_t h, vid_t v) {
    if (bv == ORD_MAX || w > bw || (w == bw && h > bh)) {
        bw = w;
        bh = h;
        bv = v;
    }
}

}  // namespace jet
