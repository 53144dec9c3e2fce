// Contraction of one level by a team of workgroups on one XCD (host side).
#pragma once
#include <hip/hip_runtime.h>

#include "arena.h"
#include "contract.h"
#include "jet_types.h"

namespace jet {

// Whether a contraction of n vertices and m edges to nc is made by a team.
bool team_contract_fits(int64_t n, int64_t m, int64_t nc);

// contract() in one launch. False when no team could start or a coarse row
// has more fine edges than the kernel's tables take: nothing is then built.
bool contract_team(const DGraph& g, const vid_t* map, vid_t nc, Arena& persist, Arena& a, hipStream_t s, Level& out);

}  // namespace jet
