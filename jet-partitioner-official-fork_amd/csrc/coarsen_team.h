// Matching of one level by a team of workgroups on one XCD (host side).
#pragma once
#include <hip/hip_runtime.h>

#include "arena.h"
#include "jet_types.h"
#include "team.h"

namespace jet {

constexpr int64_t TEAM_MATCH_M = 1000000;  // edges of a level the kernel takes at most

// Whether the calling thread's level of n vertices and m edges is matched by
// a team.
bool team_match_fits(int64_t n, int64_t m);

// coarsen_match in one launch; returns nc, or -1 when no team could start
// (`map` is then untouched).
int32_t coarsen_match_team(const DGraph& g, bool uniform, uint64_t seed, int32_t level, bool two_hop, vid_t* map,
                           Arena& a, hipStream_t s);

}  // namespace jet
