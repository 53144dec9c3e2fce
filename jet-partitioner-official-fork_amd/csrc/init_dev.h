// One coarsening level of the initial partitioner's hierarchy on the device.
#pragma once
#include <vector>

#include "arena.h"
#include "contract.h"
#include "jet_types.h"

namespace jet {

// The level that jet_init::init_hierarchy's step `lvl` makes of g on the host
// (handshake matching, leftover pairs, rows in first-seen order), for graphs
// of at least jet_init::PAR_MATCH_EDGES entries. vw: g's vertex weights on the
// host; receives the coarse level's. The arrays come from persist. Returns
// false (nothing allocated) when the level shrinks by less than 10%: the
// hierarchy ends with g.
bool init_coarsen_device(const DGraph& g, std::vector<int32_t>& vw, uint64_t seed, int lvl, Arena& persist, Arena& a,
                         hipStream_t s, Level& out);

}  // namespace jet
