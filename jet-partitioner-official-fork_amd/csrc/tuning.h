// Launch-shape and path parameters that do not change results (every setting
// gives the same partition): process-wide, read from the device's tuning
// table at context creation, settable through jet_tuning_set (the autotuner
// and the tests use it).
#pragma once
#include <cstdint>
#include <string>

namespace jet {

struct Tuning {
    // levels of up to this many vertices (at most 65536, 256 parts, and not
    // too many edges: team_fits) are refined in one launch by a team of
    // workgroups on one XCD (0: never)
    int64_t wg_max_n = 65536;
    // once the levels that jobs of the batched and served layer refined by one
    // workgroup each; that path is closed (a case with levels of up to 16384
    // vertices ended in a GPU fault of unknown cause), and the value is kept so
    // that tables and callers that set it still work, but read by nothing
    int64_t batch_wg_max_n = 0;
    // in the team's kernel, candidates and moves of higher degree are taken by a
    // whole wave instead of a group of lanes
    int64_t wg_big_deg = 32;
    // polls of a team's first workgroup before it gives up waiting for the
    // others (some 0.1 s; 0: every team of more than one workgroup is given up)
    int64_t team_start_spins = 1 << 18;
    // iterations of a level that one launch of a team runs at most
    int64_t team_launch_iters = 1 << 16;
    // "small" levels: every connectivity row is built by a wave, the
    // afterburner takes ab_lanes_small times its lanes per candidate, and the
    // rebalancers' select kernels run 128-thread workgroups
    int64_t small_level_n = 32768;
    int64_t ab_lanes_small = 2;
    // lanes per move in the update passes: upd_lanes times the level's lane
    // group (from its average degree), at most a wave
    int64_t upd_lanes = 2;
    // candidates of degree above 128 times this are taken by a whole workgroup,
    // moves in slices of 1024 edges (of degree above 64 by a wave)
    int64_t upd_big_slices = 16;
    // levels of up to this many vertices run LP select with one pass per wave
    int64_t lp_one_pass_n = 524288;
    // contraction: coarse rows of up to ct_wave_max fine entries take the
    // one-wave LDS table (256 slots), up to ct_block_max the one-workgroup
    // table (8192 slots), longer rows the radix spill path
    int64_t ct_wave_max = 128;
    int64_t ct_block_max = 4096;
    // strong rebalancing: up to this many re-drawn vertices are put in id
    // order in LDS, longer lists in global memory
    int64_t redraw_lds_max = 8192;
    // rebalancers' select kernels: at most this many workgroups (each a
    // contiguous range of vertices)
    int64_t sel_max_blocks = 1024;
    // and flush their bucket maps into one copy of the bucket array per this
    // many workgroups (at most 16 copies; up to 64 parts, per at most 32 to 64:
    // Refiner::rebalance)
    int64_t sel_copy_wgs = 256;
};

Tuning& tuning();
// Contexts of at least this many workers hold their jobs' teams to
// TEAM_BATCH_N vertices (team.h); jobs of smaller ones run as single calls do.
constexpr int BATCH_MANY_WORKERS = 8;
// Applies a tuning table (lines "name value"; '#' starts a comment). Returns
// the number of settings applied, or -1 when the file cannot be read or holds
// an unknown name or a value out of range (nothing is applied then).
int tuning_load(const std::string& path);

// Loads the table for the device architecture `arch` (e.g. "gfx950") once per
// process: $JET_TUNING_FILE when set, else tuning/<arch>.txt beside the
// library. Parameters already set through jet_tuning_set keep their values.
void tuning_init_once(const std::string& arch);

}  // namespace jet
