// Whole-level refinement by a team of workgroups on one XCD (host side).
#pragma once
#include <hip/hip_runtime.h>

#include "jet_types.h"
#include "team.h"

namespace jet {

constexpr int64_t TEAM_MAX_M = 600000;
constexpr int32_t TEAM_MAX_K = 256;
constexpr int32_t TEAM_MAX_NBK = 16384;
constexpr int TEAM_MAX_TEMPS = 20;

// Controller state of jet_refine (jet_refiner.hpp:1079-1134).
struct LevelState {
    int64_t curr_cut, curr_imb, best_cut, best_imb;
    int32_t temp_idx, count, balance_counter, iterations, lp_iterations;
    int32_t changed, status;
};

// Device words the level's team shares: the team's own, and the step's sums.
struct RefineCtl {
    TeamCtl team;
    int32_t moves[2], ranked, redraws, err, max_deg, pad4[26];
    int64_t cut[2], pad5[14];
};

struct TeamParams {
    DGraph g;
    int32_t k, sections, nbk;
    int32_t big_deg;  // items of higher degree are taken by a whole wave
    int32_t lanes;    // lanes per smaller item: a power of two up to a wave
    int32_t team;     // workgroups wanted
    int32_t xcd;      // the XCD they run on
    int32_t start_spins;
    int32_t own;      // consecutive vertices of a workgroup's chunks (launch_refine_team sets it)
    int64_t opt, size_max, imb_max, max_dest_weak, max_dest_strong;
    double tol;
    int32_t ntemps;
    double temps[TEAM_MAX_TEMPS];
    LevelState start;
    int32_t resume;     // the level goes on from `start` (LEVEL_MORE); else from best_part
    int32_t iter_cap;   // iterations of the level after which the launch ends
    part_t* part;
    part_t* best_part;  // in: the level's partition; out: the best one
    int2* conn;         // m slots: the table of row i starts at slot rowptr[i]
    int32_t* conn_size;
    part_t* dest_cache;
    int32_t* lock;
    int32_t* gain_p;
    int32_t* pregain;
    part_t* dest;
    int32_t* bid;
    int32_t* stamp;
    int32_t gen0;  // the level's steps stamp gen0 + 1, gen0 + 2, ...
    int32_t* mark;     // n zeros
    int64_t* score;    // n
    uint64_t* rkey;    // n
    int32_t* rweight;  // n
    vid_t* redraw;     // n
    int32_t* buckets;  // nbk + 1 zeros
    int64_t* sizes;
    int64_t* best_sizes;
    int64_t* evict_adjust;
    RefineCtl* ctl;
    int64_t* host_out;  // TEAM_OUT_WORDS mapped host words, then the sequence word
    int64_t seq;
};

// Best cut, best imbalance, current cut, current imbalance; then pairs of 32
// bits (low, high): iterations and LP iterations, error bits and balance
// counter, and in 16 bits each status, changed, temperature, count. With the
// sequence word they fill one 64-byte line: the host has seen words of another
// line older than the sequence word written after them, in spite of the fence
// between (one in some 300 batches of 24 graphs; none with one line).
constexpr int TEAM_OUT_WORDS = 7;
constexpr int TEAM_MAILBOX = 16;  // their place in the thread's mailbox
static_assert(TEAM_MAILBOX % 8 == 0 && TEAM_OUT_WORDS < 8, "one 64-byte line");
// Levels of more edges are refined by a team only when no row is longer.
constexpr int64_t TEAM_REGULAR_M = 100000;
constexpr int32_t TEAM_MAX_DEG = 128;

// Whether a level fits the team kernel's limits.
bool team_fits(int64_t n, int64_t m, int32_t k, int64_t nbk, int64_t max_n);
// Workgroups for a level of n vertices and m edges.
int32_t team_size(int64_t n, int64_t m);
// Clears the control words and the bucket sums and copies the best part sizes
// to the current ones, then runs the level, on stream s. The result words are
// published to p.host_out; status LEVEL_ABANDONED (or a finished stream without
// a result) means that no team could start: the level's arrays are untouched.
// LEVEL_IRREGULAR: the level has rows of more than TEAM_MAX_DEG edges, and too
// many edges (likewise nothing has changed). LEVEL_MORE: iter_cap was reached;
// a launch with `resume` and the published state goes on.
enum : int32_t { LEVEL_DONE = 0, LEVEL_MORE = 1, LEVEL_STALLED = 2, LEVEL_ABANDONED = 3, LEVEL_IRREGULAR = 4 };
void launch_refine_team(TeamParams p, hipStream_t s);

}  // namespace jet
