// Host initial partitioner (csrc/initpart.cpp): the C entry point for the
// coarsest graph, and the coarsening hierarchy it uses for large graphs.
#pragma once
#include <cstdint>
#include <vector>

extern "C" int jet_host_initpart(int32_t n, const int64_t* xadj, const int32_t* adj, const int32_t* adjw,
                                 const int32_t* vw, int32_t k, double imb, uint64_t seed, int32_t* part);

namespace jet_init {

// One coarser level of the initial partitioner's hierarchy.
struct HostLevel {
    int32_t n = 0;
    std::vector<int64_t> xadj;
    std::vector<int32_t> adj, adjw, vw;
    std::vector<int32_t> map;  // vertex of the next finer level -> vertex of this level
};

// Coarsest graphs with at least this many adjacency entries are partitioned
// multilevel k-way: coarsened further on the host (init_hierarchy), the
// smallest level partitioned by jet_host_initpart, and the partition refined
// back up with Jet refinement level by level (the structure of METIS's k-way
// scheme, with Jet as its refiner).
constexpr int64_t INIT_ML_EDGES = int64_t(1) << 20;

inline bool wants_hierarchy(int32_t n, int64_t m, int32_t k) {
    return m >= INIT_ML_EDGES && (int64_t)n > 8 * (int64_t)k;
}

// Caps the host threads that the initial partitioner uses for calls made on
// the calling thread (0: no cap). Results do not depend on the thread count.
void set_thread_budget(int threads);

// The levels coarser than the graph (first = one level coarser), down to
// about max(1000, 8 k) vertices or until a level shrinks by less than 10%.
// first_lvl: the levels already made (on the device) of the hierarchy.
std::vector<HostLevel> init_hierarchy(int32_t n, const int64_t* xadj, const int32_t* adj, const int32_t* adjw,
                                      const int32_t* vw, int32_t k, uint64_t seed, int first_lvl = 0);

// ---- the hierarchy's rules, for the device's coarsening of large levels
// Graphs of at least this many entries are matched by handshakes, in this many
// rounds (smaller ones in a seeded order, one vertex after another).
constexpr int64_t PAR_MATCH_EDGES = int64_t(1) << 21;
constexpr int HANDSHAKE_ROUNDS = 6;
constexpr int MAX_LEVELS = 64;
int32_t hierarchy_target(int32_t k);                 // levels of at most this many vertices end it
uint64_t level_seed(uint64_t seed, int lvl);         // seed of level lvl's matching
int64_t match_weight_cap(int64_t total_w);           // heaviest matched pair
bool shrinks_enough(int32_t nc, int32_t n);

// What the matching leaves (mate[v] < 0) paired: leaves sharing their first
// neighbour (first_adj, -1: no neighbour), and isolated vertices; then the
// coarse ids, in order of first member, with each coarse vertex's members and
// weight.
struct CoarseMap {
    int32_t n = 0;
    std::vector<int32_t> map, first, second, vw;  // second -1: one member
};
CoarseMap finish_matching(int32_t n, std::vector<int32_t>& mate, const int32_t* first_adj, const int32_t* vw,
                          int64_t cap);

}  // namespace jet_init
